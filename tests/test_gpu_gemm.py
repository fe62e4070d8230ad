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


# (rows, inputs, tokens): 64 x 128 tiles; 128 x 128; 256 x 256 where bf16 x takes it
SHAPES = [(6912, 256, 65), (6912, 2560, 130), (300, 208, 3300), (2049, 80, 1100), (129, 16, 8200),
          (1000, 80, 6200), (2049, 64, 5800), (6912, 272, 2000)]


@pytest.mark.parametrize("M,K,B", SHAPES)
@pytest.mark.parametrize("kind", ["bf16", "bf16_x", "fp32"])
def test_prefill_shapes(pkg, dev, M, K, B, kind):
    """One product (bf16 x and codebook), two (bf16 x, fp32 codebook), three (fp32 x)."""
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
    """Tokens of very different size (each has its own scale), all-zero tokens, one value 10^4
    times the others; a codebook of tiny values, and one whose unused centroid is 10^9 times the
    used ones (too wide for its half pieces: the batched kernel).  Error per token, relative to
    the token's largest output."""
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
