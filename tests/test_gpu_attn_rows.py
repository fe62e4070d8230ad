"""GPU parity of the many-row streamed attention (attn_rows_kernel) with fp64: every tile type and
head dim it takes, ragged rows and tokens, causal offsets, rows that see nothing, runs merged
from partials and runs that continue the state, int8 pages.

Bar: 1e-12 relative to the largest |out| for fp64 queries (the arithmetic is fp64), the output
type's rounding otherwise."""
import numpy as np
import pytest

from oracle import numpy_oracle as no

pytestmark = pytest.mark.gpu


def want(q, k, v, causal, start):
    """[B, H, S, D] fp64 attention per head, k and v grouped."""
    q, k, v = (t.double().cpu().numpy() for t in (q, k, v))
    R = q.shape[1] // k.shape[1]
    out = np.empty(q.shape)
    for b in range(q.shape[0]):
        K, V = (np.repeat(t[b], R, axis=0) for t in (k, v))
        s = np.einsum("hsd,htd->hst", q[b], K) / np.sqrt(q.shape[-1])
        if causal:
            hide = np.arange(K.shape[1])[None, :] > start + np.arange(q.shape[2])[:, None]
            s = np.where(hide[None], -np.inf, s)
        m = s.max(-1, keepdims=True)
        p = np.exp(s - np.where(np.isinf(m), 0, m))
        l = p.sum(-1, keepdims=True)
        out[b] = np.einsum("hst,htd->hsd", p / np.where(l > 0, l, 1), V)
    return out


# (batch, query heads, kv heads, queries, tokens, causal, start)
SHAPES = [(1, 32, 8, 70, 1111, True, 1041),     # 280 rows: a last block of 24; ragged tiles
          (2, 8, 8, 65, 2050, True, 100),       # rows cross no head boundary; most tokens hidden
          (1, 16, 2, 33, 4100, False, 0),       # a block of 64 rows over two heads
          (1, 16, 16, 300, 600, True, 300)]     # 80 row blocks x 2: several runs per block


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("D,dt", [(128, "bfloat16"), (64, "float32"), (80, "float16"), (128, "float64"),
                                  (64, "float64"), (128, "float32")])
def test_forward(pkg, dev, shape, D, dt):
    import torch
    B, Hq, Hk, S, T, causal, start = shape
    g = torch.Generator().manual_seed(S + T + D)
    dtype = getattr(torch, dt)
    q = torch.randn(B, Hq, S, D, generator=g).to(dtype).to(dev)
    k, v = (torch.randn(B, Hk, T, D, generator=g).to(dtype).to(dev) for _ in range(2))
    att = pkg.long_context.OnlineSoftmaxBlockAttention(Hq, Hk, D, causal=causal)
    out = att.forward(q, k, v, query_start_pos=start)
    ref = want(q, k, v, causal, start)
    got = out.double().cpu().numpy()
    tol = {"float64": 1e-12, "float32": 1e-6, "float16": 2e-3, "bfloat16": 1e-2}[dt]
    assert np.abs(got - ref).max() <= tol * np.abs(ref).max()


@pytest.mark.parametrize("S,start", [(64, 4000), (100, -1), (256, 2000)])
def test_int8_pages(pkg, dev, S, start):
    """Pages of 48 tokens (steps of 32 and 16), the last one partial; rows before the first token
    see nothing and give zero."""
    import torch
    Hq, Hk, D, T = 32, 8, 128, 4099
    g = torch.Generator().manual_seed(S)
    cache = pkg.long_context.PagedCompressedKVCache(48, max_resident_pages=128, sink_pages=2)
    cache.append(*(torch.randn(1, Hk, T, D, generator=g).to(dev) for _ in range(2)))
    pages = list(cache.iter_dequantized_pages(torch.float64))
    k, v = (torch.cat([p[i] for p in pages], 2) for i in (0, 1))
    q = torch.randn(1, Hq, S, D, generator=g, dtype=torch.float64).to(dev)
    att = pkg.long_context.OnlineSoftmaxBlockAttention(Hq, Hk, D, causal=True)
    out, rep = att.forward_stream(q, cache, query_start_pos=start)
    ref = want(q, k, v, True, start)
    assert np.abs(out.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max()
    if start < 0:
        assert not out[:, :, 0].any()
    assert rep.kv_tokens == T


def test_state_continues_over_updates(pkg, dev):
    """Three streamed tiles, the middle one small (the other kernel), fold into one state."""
    import torch
    Hq, Hk, S, D = 32, 8, 128, 128
    g = torch.Generator().manual_seed(4)
    q = torch.randn(1, Hq, S, D, generator=g, dtype=torch.float64).to(dev)
    tiles = [tuple(torch.randn(1, Hk, n, D, generator=g, dtype=torch.float64).to(dev) for _ in range(2))
             for n in (1500, 40, 2000)]
    att = pkg.long_context.OnlineSoftmaxBlockAttention(Hq, Hk, D, causal=True)
    out, rep = att.forward_stream(q, tiles, query_start_pos=3300)
    k, v = (torch.cat([t[i] for t in tiles], 2) for i in (0, 1))
    ref = want(q, k, v, True, 3300)
    assert np.abs(out.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max()
    assert rep.kv_tokens == 3540


def test_strided_tensors_and_extremes(pkg, dev):
    """Transposed [B, S, H, D] storage; scores far apart, one +inf value in v and all-equal scores."""
    import torch
    B, Hq, Hk, S, T, D = 1, 16, 4, 64, 2048, 64
    g = torch.Generator().manual_seed(6)
    q = (torch.randn(B, S, Hq, D, generator=g) * 30).to(dev).transpose(1, 2)
    k = (torch.randn(B, T, Hk, D, generator=g) * 30).to(dev).transpose(1, 2)
    v = torch.randn(B, T, Hk, D, generator=g).to(dev).transpose(1, 2)
    att = pkg.long_context.OnlineSoftmaxBlockAttention(Hq, Hk, D, causal=False)
    out = att.forward(q.double(), k, v)
    ref = want(q, k, v, False, 0)
    assert np.abs(out.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max()
    out = att.forward(torch.zeros_like(q).double(), k, v)
    assert np.abs(out.cpu().numpy() - want(torch.zeros_like(q), k, v, False, 0)).max() <= 1e-12
    v = v.clone()
    v[0, 1, 77, 5] = float("inf")
    out = att.forward(torch.zeros_like(q), k, v)
    bad = torch.isinf(out)
    assert bad[0, 4:8, :, 5].all() and int(bad.sum()) == 4 * S


@pytest.mark.parametrize("causal", [True, False])
def test_more_rows_than_one_update_takes(pkg, dev, causal):
    """600000 queries of one head of 16 dims: more than an update's 65535 blocks of 8 rows."""
    import torch
    S, T, D = 600000, 40, 16
    g = torch.Generator().manual_seed(8)
    q = torch.randn(1, 1, S, D, generator=g).to(dev)
    k, v = (torch.randn(1, 1, T, D, generator=g).to(dev) for _ in range(2))
    att = pkg.long_context.OnlineSoftmaxBlockAttention(1, 1, D, q_block_size=4096, causal=causal)
    out = att.forward(q, k, v)
    rows = [0, 1, T - 1, 4095, 4096, 524279, 524280, S - 1]
    for r in rows:
        ref = want(q[:, :, r:r + 1], k, v, causal, r)
        assert np.abs(out[:, :, r:r + 1].cpu().numpy() - ref).max() <= 1e-6 * np.abs(ref).max(), r


# (query heads, kv heads, queries, tokens, start, head dim)
HIDDEN = [(4, 4, 300, 300, 0, 32), (4, 2, 301, 301, 0, 96), (4, 4, 300, 500, 200, 256), (4, 1, 75, 75, 0, 64),
          (2, 2, 7, 700, 500, 128),
          # attn_rows_kernel: one head per row block; two; every step seen in part by some
          (16, 16, 300, 600, 300, 128), (32, 8, 70, 1111, 1041, 64), (32, 8, 130, 1500, 1370, 80),
          (16, 4, 512, 2048, 1536, 128)]


@pytest.mark.parametrize("shape", HIDDEN)
@pytest.mark.parametrize("dt", ["float64", "bfloat16"])
def test_hidden_values_reach_no_result(pkg, dev, shape, dt):
    """A NaN and an inf row of v change exactly the queries that see them: row blocks over two
    heads, and tokens that all rows of a block see, some, or none."""
    import torch
    Hq, Hk, S, T, start, D = shape
    g = torch.Generator().manual_seed(D + S)
    dtype = getattr(torch, dt)
    q = torch.randn(1, Hq, S, D, generator=g).to(dtype).to(dev)
    k, v = (torch.randn(1, Hk, T, D, generator=g).to(dtype).to(dev) for _ in range(2))
    att = pkg.long_context.OnlineSoftmaxBlockAttention(Hq, Hk, D, causal=True)
    ref = want(q, k, v, True, start)
    tol = {"float64": 1e-12, "bfloat16": 1e-2}[dt] * np.abs(ref).max()
    assert np.abs(att.forward(q, k, v, query_start_pos=start).double().cpu().numpy() - ref).max() <= tol
    first = S // 2 + 1                                # the first query that sees the NaN
    v[:, :, start + first] = float("nan")
    v[:, :, start + S - 1] = float("inf")
    out = att.forward(q, k, v, query_start_pos=start).double().cpu().numpy()
    assert np.abs(out[:, :, :first] - ref[:, :, :first]).max() <= tol
    assert np.isnan(out[:, :, first:]).all()


def test_infinite_value_in_a_partial_step(pkg, dev):
    """attn_rows_kernel: +inf in the last value row of a step that is not full stays inf."""
    import torch
    q, k = torch.zeros(1, 16, 64, 64, device=dev), torch.zeros(1, 4, 2050, 64, device=dev)
    v = torch.ones(1, 4, 2050, 64, device=dev)
    v[:, 2, -1, 5] = float("inf")
    out = pkg.long_context.OnlineSoftmaxBlockAttention(16, 4, 64, causal=False).forward(q, k, v)
    assert torch.isinf(out[:, 8:12, :, 5]).all()
    out[:, 8:12, :, 5] = 1
    assert (out - 1).abs().max() < 1e-6
