"""GPU parity of the math engine's MFMA kernel (lut_rvq_mm_kernel) with the fp64 dense product:
block sizes 4 and multiples of 8, every code width, up to four stages, ragged rows, columns and
tokens, unaligned inputs, and infinite and NaN values.

Bars as in test_gpu_rvq: rel <= 1e-5 (max-abs error / max |ref|) for fp32 inputs, <= 1e-2 for
bf16; bit-exact on integers."""
import numpy as np
import pytest

from conftest import rel_err
from oracle import gen
from oracle import numpy_oracle as no
from test_gpu_rvq import make_encoded

pytestmark = pytest.mark.gpu


def dense(cbs, packed, bits, rows, cols, block, scales):
    G = -(-cols // block)
    W = sum(cbs[s].astype(np.float64)[no.unpack_codes(packed[s], bits, rows * G).reshape(rows, G)]
            for s in range(len(cbs)))
    return W.reshape(rows, G * block)[:, :cols] * scales.astype(np.float64)[:, None]


@pytest.mark.parametrize("rows,cols,block,bits,stages", [
    (33, 1003, 8, 4, 2),       # odd columns: every row at another alignment
    (70, 100, 4, 2, 3),        # block 4: two codes per read, a last chunk half full
    (300, 250, 24, 1, 2),      # block 24: chunks across groups
    (31, 17, 64, 8, 1),        # one partial chunk of one group
    (257, 2048, 32, 8, 2),     # 96 KB of codebook pieces
    (4100, 48, 16, 8, 4),      # three chunks for eight waves; two token tiles per workgroup
    (65, 999, 40, 4, 1),
])
@pytest.mark.parametrize("B", [3, 32, 33, 64, 129])
@pytest.mark.parametrize("bf16", [False, True])
def test_matches_fp64(pkg, dev, rows, cols, block, bits, stages, B, bf16):
    import torch
    me = pkg.math_engine
    enc, cbs, packed, scales = make_encoded(me, torch, dev, rows, cols, block, bits, stages,
                                            seed=rows + cols + B)
    r = gen.rng(B)
    x = torch.from_numpy(r.normal(size=(B, cols)).astype(np.float32))
    bias = r.normal(size=rows).astype(np.float32)
    if bf16:
        x = x.bfloat16()
    # an input that starts one element past an aligned address
    buf = torch.empty(B * cols + 1, dtype=x.dtype, device=dev)
    xd = buf[1:].view(B, cols)
    xd.copy_(x)
    y = me.subspace_lut_rvq_gemm(xd, enc, torch.from_numpy(bias).to(dev)).float().cpu().numpy()
    want = x.double().numpy() @ dense(cbs, packed, bits, rows, cols, block, scales).T + bias
    assert rel_err(y, want) < (1e-2 if bf16 else 1e-5)


@pytest.mark.parametrize("block,bits,stages", [(8, 4, 3), (16, 8, 2), (4, 4, 2), (24, 2, 2)])
def test_integers_bit_exact(pkg, dev, block, bits, stages):
    import torch
    me = pkg.math_engine
    rows, cols, B = 300, 1000, 40
    enc, cbs, packed, scales = make_encoded(me, torch, dev, rows, cols, block, bits, stages, seed=3,
                                            integer=True)
    x = gen.rng(4).integers(-4, 5, size=(B, cols)).astype(np.float32)
    y = me.subspace_lut_rvq_gemm(torch.from_numpy(x).to(dev), enc).cpu().numpy()
    want = x.astype(np.float64) @ dense(cbs, packed, bits, rows, cols, block, scales).T
    assert np.array_equal(y, want.astype(np.float32))


def test_infinities_and_nan(pkg, dev):
    """An infinite x, a NaN, values near the largest float and an infinite centroid give what
    plain fp32 sums give; the other tokens and rows stay exact."""
    import torch
    me = pkg.math_engine
    rows, cols, B = 64, 64, 8
    enc, cbs, packed, scales = make_encoded(me, torch, dev, rows, cols, 16, 8, 1, seed=8)
    codes = enc.codes(0).view(rows, 4)
    codes[:, 0] = codes[:, 0].clamp(min=1)
    codes[5, 2] = 0                                   # only row 5 (and rows that drew it) use centroid 0
    enc.packed_codes[0] = me.pack_codes(codes, 8)
    enc.codebooks[0, 0, 3] = float("inf")
    x = torch.from_numpy(gen.rng(9).normal(size=(B, cols)).astype(np.float32)).to(dev)
    x[1, 7] = float("inf")
    x[2, 9] = float("-inf")
    x[3, 20] = float("nan")
    x[4, 30] = 3.4e38
    y = me.subspace_lut_rvq_gemm(x, enc)
    W = (enc.codebooks[0][codes.long()].flatten(1) * enc.row_scales[:, None]).double()
    plain = (enc.codebooks[0][codes.long()].flatten(1))
    want = (x.double() @ plain.double().T).float() * enc.row_scales
    # token 4's sums pass the largest fp32 value in fp32 but not in the fp64 of `want`, so where it
    # meets the infinite centroid the fp32 result may be inf - inf: any non-finite value is right
    inf_rows = torch.isinf(plain).any(1)
    assert not torch.isfinite(y[4, inf_rows]).any()
    y[4, inf_rows] = want[4, inf_rows]
    same = torch.isfinite(want)
    assert torch.equal(torch.isfinite(y), same)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    assert torch.equal(y[torch.isinf(want)], want[torch.isinf(want)])
    err = ((y - want).abs()[same] / (x.abs().double() @ W.abs().T).float()[same]).max()
    assert float(err) < 1e-5
