"""GPU parity of the prefill-batch LUT linear (lut_gemm.hip) against fp64, through the C-ABI:
every tile shape and product kind, ragged rows, tokens and input slices, outlier groups (empty
rows, rows of more than four groups, dense rows), and the calls that must stay on the batched
kernel.

Bars: bit-exact on integer inputs (every partial sum exact); rel <= 1e-5 (max-abs error /
max |ref|) for fp32, <= 1e-2 for bf16 activations, as in test_gpu_linear.
"""
import ctypes

import numpy as np
import pytest

from conftest import rel_err
from oracle import gen
from oracle import numpy_oracle as no

pytestmark = pytest.mark.gpu


def handle(pkg, d, M, K):
    nat = pkg.native.NativeSplitManifoldLinear(K, M, 16, 256)
    nat.initialize_weights(d["codebook"], d["codes"], d["scales"], d.get("bias"))
    if d.get("csr") is not None:
        nat.set_outliers(*d["csr"])
    return nat


def forward(pkg, nat, x):
    import torch
    y = torch.empty(x.shape[0], nat.out_features, device=x.device, dtype=x.dtype)
    rc = pkg.lib().ojasx_linear_forward_device(
        nat.handle, ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(y.data_ptr()), x.shape[0],
        0 if x.dtype == torch.float32 else 1, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, pkg.lib().ojasx_get_last_error()
    return y


def to_bf16(a):
    import torch
    return torch.from_numpy(a).bfloat16().float().numpy()


def make(M, K, B, seed, density=0.0038, cb_bf16=False, x_bf16=False):
    d = gen.linear(M, K, B=B, seed=seed, scales="u", bias=True, density=density)
    if cb_bf16:
        d["codebook"] = to_bf16(d["codebook"])
    if x_bf16:
        d["x"] = to_bf16(d["x"])
    return d


def reference(d, rows=None):
    x = d["x"] if rows is None else d["x"][rows]
    return no.linear_fp64(x, d["codebook"], d["codes"], d["scales"], d["bias"], d["csr"])


# (rows, inputs, tokens): every tile shape of each product kind among them
SHAPES = [(6912, 256, 65), (6912, 2560, 130), (300, 208, 3300), (2049, 80, 1100), (129, 16, 8200),
          (1000, 80, 6200), (2049, 64, 5800), (6912, 272, 2000)]


@pytest.mark.parametrize("M,K,B", SHAPES)
@pytest.mark.parametrize("kind", ["bf16", "bf16_x", "fp32"])
def test_prefill_shapes(pkg, dev, M, K, B, kind):
    """One product (bf16 x and codebook), three (bf16 x, fp32 codebook), six (fp32 x)."""
    import torch
    d = make(M, K, B, M + K + B, cb_bf16=kind == "bf16", x_bf16=kind != "fp32")
    nat = handle(pkg, d, M, K)
    x = torch.from_numpy(d["x"]).to(dev)
    y = forward(pkg, nat, x if kind == "fp32" else x.bfloat16()).float().cpu().numpy()
    # tokens at the edges of the tiles and a few between
    rows = sorted({0, 1, 31, 32, 63, 64, B // 2, B - 33, B - 2, B - 1} & set(range(B)))
    assert rel_err(y[rows], reference(d, rows)) < (1e-5 if kind == "fp32" else 1e-2)
    # the other tokens: against the same call's batched kernel, 64 tokens at a time
    # (64 tokens never take the tiles under test)
    parts = [forward(pkg, nat, (x if kind == "fp32" else x.bfloat16())[b:b + 64].contiguous())
             for b in range(0, B, 64)]
    assert rel_err(y, torch.cat(parts).float().cpu().numpy()) < (1e-5 if kind == "fp32" else 1e-2)


@pytest.mark.parametrize("kind", ["bf16", "fp32"])
@pytest.mark.parametrize("M,K,B", [(333, 2000, 4000), (6912, 464, 260)])
def test_integer_bit_exact(pkg, dev, M, K, B, kind):
    """Integers and outliers whose sums are exact in fp32: any order gives these bits; in bf16
    the exact sum rounded once."""
    import torch
    r = np.random.default_rng(M + B)
    d = dict(codebook=r.integers(-4, 5, size=(256, 16)).astype(np.float32),
             codes=r.integers(0, 256, size=(M, K // 16)).astype(np.uint8),
             scales=r.choice([0.5, 1.0, 2.0], size=M).astype(np.float32), bias=None,
             x=r.integers(-3, 4, size=(B, K)).astype(np.float32))
    rp, cl, vl = gen.csr_outliers(r, M, K, density=0.01)
    d["csr"] = (rp, cl, r.integers(-20, 21, size=vl.size).astype(np.float32))
    nat = handle(pkg, d, M, K)
    W = no.dequantize(d["codebook"], d["codes"], d["scales"], csr=d["csr"])
    want = torch.from_numpy(d["x"].astype(np.float64) @ W.T)
    x = torch.from_numpy(d["x"]).to(dev)
    if kind == "fp32":
        assert torch.equal(forward(pkg, nat, x).cpu(), want.float())
    else:
        assert torch.equal(forward(pkg, nat, x.bfloat16()).cpu(), want.float().bfloat16())


@pytest.mark.parametrize("kind", ["bf16", "fp32"])
def test_outlier_groups(pkg, dev, kind):
    """Rows with 0, 1, 3, 4, 5, 64, 65 and 200 outliers, a first and a last row without any."""
    import torch
    M, K, B = 2100, 512, 1100
    d = make(M, K, B, 5, cb_bf16=kind == "bf16", x_bf16=kind == "bf16")
    r = np.random.default_rng(1)
    counts = r.choice([0, 0, 1, 3, 4, 5, 8, 64, 65, 200], size=M)
    counts[[0, -1]] = 0
    cols = np.concatenate([np.sort(r.choice(K, size=n, replace=False)) for n in counts]).astype(np.int32)
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    d["csr"] = (rp, cols, r.normal(size=cols.size).astype(np.float32))
    nat = handle(pkg, d, M, K)
    x = torch.from_numpy(d["x"]).to(dev)
    y = forward(pkg, nat, x if kind == "fp32" else x.bfloat16()).float().cpu().numpy()
    rows = [0, 5, 64, 500, B - 1]
    assert rel_err(y[rows], reference(d, rows)) < (1e-5 if kind == "fp32" else 1e-2)
    nat.set_outliers(np.zeros(M + 1, np.int32), np.zeros(0, np.int32), np.zeros(0, np.float32))
    d["csr"] = None
    y = forward(pkg, nat, x if kind == "fp32" else x.bfloat16()).float().cpu().numpy()
    assert rel_err(y[rows], reference(d, rows)) < (1e-5 if kind == "fp32" else 1e-2)


def test_scales_of_tokens_and_codebook(pkg, dev):
    """Tokens of very different size, all-zero tokens, one value 10^4 times the others; a codebook
    of tiny values, and one whose unused centroid is 10^9 times the used ones.  Error per token,
    relative to the token's largest output."""
    import torch
    M, K, B = 6912, 512, 260
    d = make(M, K, B, 9)
    d["bias"] = None
    d["x"] *= np.exp2(np.random.default_rng(2).integers(-40, 41, size=(B, 1))).astype(np.float32)
    d["x"][7] = 0
    d["x"][11, 3] *= 1e4
    for case in ("plain", "tiny", "wide"):
        if case == "tiny":
            d["codebook"] = d["codebook"] * np.float32(2.0 ** -60)
        elif case == "wide":
            d["codebook"] = d["codebook"] * np.float32(2.0 ** 60)
            d["codebook"][0] = 2e7
            d["codes"] = np.maximum(d["codes"], 1)
        nat = handle(pkg, d, M, K)
        y = forward(pkg, nat, torch.from_numpy(d["x"]).to(dev)).cpu().numpy()
        want = reference(dict(d, bias=np.zeros(M, np.float32)))
        top = np.abs(want).max(1, keepdims=True)
        assert not y[7].any()
        assert (np.abs(y - want) / np.where(top > 0, top, 1)).max() < 1e-5, case


@pytest.mark.parametrize("bf16_x", [False, True])
@pytest.mark.parametrize("wide", ["x", "codebook"])
def test_wide_range_inside_a_token(pkg, dev, wide, bf16_x):
    """One value of a token 1 to 3e38 times the others in a place where a third of the rows have
    a zero centroid and a third a centroid that is zero in that dim alone; and a codebook whose
    dims 8 .. 15 are 1 to 3e-30 times dims 0 .. 7, with x zero in dims 0 .. 7.  Both are products
    of ordinary size for those rows, held as if the large values were not there: the error
    against 64 bits, relative to the token's largest output over those rows, is that of fp32 sums
    (3e-7; the exact pieces leave 2^-22 of a term and sums of 96 rounded terms), plus the output's
    own rounding in bf16 (8 significant bits to nearest: 2^-8 of the value)."""
    import torch
    M, K, B, dim = 6912, 512, 320, 16 * 5 + 3
    d = make(M, K, B, 21, density=0.0, x_bf16=bf16_x)
    d["bias"], d["csr"] = None, None
    d["codebook"][0] = 0
    d["codebook"][1, dim % 16] = 0
    d["codes"] = np.maximum(d["codes"], 2)
    rows = np.arange(M) % 3 < 2                       # the rows that do not see the large values
    if wide == "x":
        d["codes"][::3, dim // 16], d["codes"][1::3, dim // 16] = 0, 1
        ratio = [1, 1e6, 1e7, 1e8, 1e10, 1e12, 1e20, 3e38]
        d["x"][:, dim] = [ratio[b % 8] for b in range(B)]
        if bf16_x:
            d["x"] = to_bf16(d["x"])
    else:
        d["x"].reshape(B, -1, 16)[:, :, :8] = 0
        rows[:] = True
    for ratio in [1] if wide == "x" else [1, 1e-6, 1e-8, 1e-12, 3e-30]:
        e = dict(d, codebook=d["codebook"].copy())
        e["codebook"][:, 8:] *= np.float32(ratio)
        nat = handle(pkg, e, M, K)
        x = torch.from_numpy(d["x"]).to(dev)
        y = forward(pkg, nat, x.bfloat16() if bf16_x else x).float().cpu().numpy()[:, rows]
        W = no.dequantize(e["codebook"], e["codes"], e["scales"])[rows]
        want = d["x"].astype(np.float64) @ W.astype(np.float64).T
        err = np.abs(y - want) - (2.0 ** -8 * np.abs(want) if bf16_x else 0)
        assert (err.max(1) / np.abs(want).max(1)).max() <= 3e-7, ratio


# tokens that take each of the tiles of three and of six products at 6912 rows
@pytest.mark.parametrize("B", [200, 512, 1024])
@pytest.mark.parametrize("case", ["bf16_second", "bf16_third", "both_nine_bits", "codebook_17_bits",
                                  "x_17_bits"])
def test_every_product_counts(pkg, dev, B, case):
    """Integers that need two or three bf16 pieces, in sums that are exact in fp32: a product left
    out or a piece read from the wrong place changes the result.  bf16 x: a pair of inputs 1 and
    -1 over centroids whose first piece is the same (and the second, for the third), so the
    result is a difference of the lower pieces, which bf16 holds.  fp32 x: four inputs per token,
    both sides of 9 to 11 bits, or one side of 17 bits and the other of at most 5."""
    import torch
    M, K = 6912, 256
    r = np.random.default_rng(B)
    i = np.arange(256)
    value = {"bf16_second": (200 << 16) + 256 * (i % 128) + 37, "bf16_third": (200 << 16) + 256 * 90 + i % 120,
             "both_nine_bits": 257 + 6 * i, "codebook_17_bits": 65793 + 257 * i, "x_17_bits": i % 31 + 1}[case]
    d = dict(codebook=np.repeat(value[:, None], 16, 1).astype(np.float32), bias=None, csr=None,
             codes=r.integers(0, 256, size=(M, K // 16)).astype(np.uint8), scales=np.ones(M, np.float32),
             x=np.zeros((B, K), np.float32))
    for b in range(B):
        at = r.choice(K // 16, size=4, replace=False) * 16 + r.integers(0, 16, size=4)
        if case.startswith("bf16"):
            d["x"][b, at[:2]] = 1, -1
        else:
            top = {"both_nine_bits": (257, 1025), "codebook_17_bits": (1, 17), "x_17_bits": (65537, 1 << 17)}[case]
            d["x"][b, at] = r.integers(*top, size=4) * r.choice([-1, 1], size=4)
    nat = handle(pkg, d, M, K)
    want = d["x"].astype(np.float64) @ no.dequantize(d["codebook"], d["codes"], d["scales"]).T
    assert np.abs(want).max() < 2 ** 24
    x = torch.from_numpy(d["x"]).to(dev)
    y = forward(pkg, nat, x.bfloat16() if case.startswith("bf16") else x)
    assert np.array_equal(y.float().cpu().numpy(), want)


def test_capture_and_streams(pkg, dev):
    """A call of the size under capture, with no call before it, and two streams at once on one
    handle from one thread: the results of an eager call."""
    import torch
    M, K, B = 6912, 512, 260
    d = make(M, K, B, 12, cb_bf16=True, x_bf16=True)
    nat = handle(pkg, d, M, K)
    xs = [torch.from_numpy(d["x"]).to(dev).bfloat16() for _ in range(2)]
    xs[1].mul_(-2)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        yg = forward(pkg, nat, xs[0])
    for _ in range(3):
        yg.zero_()
        g.replay()
        want = forward(pkg, nat, xs[0])
        torch.cuda.synchronize()
        assert rel_err(yg.float().cpu().numpy(), want.float().cpu().numpy()) < 1e-2
    side = [torch.cuda.Stream(), torch.cuda.Stream()]
    eager = [forward(pkg, nat, x) for x in xs]
    torch.cuda.synchronize()
    got = [None, None]
    for _ in range(4):
        for i in (0, 1):
            with torch.cuda.stream(side[i]):
                got[i] = forward(pkg, nat, xs[i])
    torch.cuda.synchronize()
    for a, b in zip(got, eager):
        assert torch.equal(a, b)


def test_eager_call_beside_a_capture(pkg, dev):
    """A handle's first prefill call (scratch and outlier groups to be allocated) on a stream of
    its own while another stream is being captured: both give the results they give alone."""
    import torch
    M, K, B = 6912, 512, 260
    d = make(M, K, B, 13, cb_bf16=True, x_bf16=True)
    nat, alone = handle(pkg, d, M, K), handle(pkg, d, M, K)
    x = torch.from_numpy(d["x"]).to(dev).bfloat16()
    y = torch.empty(B, M, device=dev, dtype=torch.bfloat16)
    want = forward(pkg, alone, x)
    side, g, a = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.zeros(64, device=dev)
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        a.add_(1)
        rc = pkg.lib().ojasx_linear_forward_device(
            nat.handle, ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(y.data_ptr()), B, 1,
            ctypes.c_void_p(side.cuda_stream))
        a.add_(1)
    assert rc == 0, pkg.lib().ojasx_get_last_error()
    torch.cuda.synchronize()
    assert torch.equal(y, want)
    for i in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert (a == 2 * (i + 1)).all()


def test_thread_ends_beside_a_capture(pkg, dev):
    """A thread that made prefill calls ends, and frees its scratch, while another thread's stream
    is being captured: the capture goes on."""
    import threading
    import torch
    M, K, B = 6912, 512, 260
    d = make(M, K, B, 14)
    nat = handle(pkg, d, M, K)
    x = torch.from_numpy(d["x"]).to(dev)
    called, end, out = threading.Event(), threading.Event(), []

    def work():
        out.append(forward(pkg, nat, x))
        torch.cuda.synchronize()
        called.set()
        end.wait(60)

    t = threading.Thread(target=work)
    t.start()
    assert called.wait(60)
    a, g = torch.zeros(64, device=dev), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g):
        a.add_(1)
        end.set()
        t.join(60)
        a.add_(1)
    assert not t.is_alive()
    for i in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert (a == 2 * (i + 1)).all()
    assert torch.equal(out[0], forward(pkg, nat, x))
