"""GPU tests of dispatch branches of the small calls: the router's two widths with ties, and the KV
append with its slots in the launch (up to 64 tokens) against the device slot mapping."""
import ctypes

import numpy as np
import pytest

from oracle import numpy_oracle as no

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E", [33, 512, 513, 1024])
@pytest.mark.parametrize("k", [1, 10, 32])
def test_router_ties_bit_exact(pkg, dev, E, k):
    """Rounded logits: many ties, some across lanes, some within one; -inf logits last."""
    import torch
    r = np.random.default_rng(E + k)
    logits = np.round(r.normal(size=(37, E)) * 4).astype(np.float32) / 4
    logits[3] = 1.0                                   # all equal
    logits[4, :E - k] = -np.inf
    idx = torch.empty(37, k, dtype=torch.int32, device=dev)
    w = torch.empty(37, k, device=dev)
    t = torch.from_numpy(logits).to(dev)
    p = lambda a: ctypes.c_void_p(a.data_ptr())
    assert pkg.lib().ojasx_moe_route_device(p(t), 37, E, k, 1, p(idx), p(w), None) == 0
    torch.cuda.synchronize()
    want_i, want_w = no.router_topk(logits, k, renorm=True)
    assert np.array_equal(idx.cpu().numpy(), want_i)
    assert np.abs(w.cpu().numpy() - want_w).max() < 1e-6


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65])
@pytest.mark.parametrize("codebook", [True, False])
def test_append_slots_in_the_launch(pkg, dev, n, codebook):
    """Caches fed n tokens at a time (64 and fewer: slots in the launch) equal one fed all at once
    through the device mapping; skipped and out-of-range slots write nothing."""
    import torch
    lc = pkg.long_context
    g = torch.Generator().manual_seed(n)
    cbs = [torch.randn(2, 256, 16, generator=g) * 40 for _ in range(2)] if codebook else [None, None]
    k, v = (torch.randn(195, 2, 64, generator=g).to(dev) for _ in range(2))
    make = lambda: lc.PagedCodeKVCache(2, 64, 16, page_size=16, max_resident_pages=64, sink_pages=1,
                                       k_codebook=cbs[0], v_codebook=cbs[1], device=dev)
    a, b = make(), make()
    a.append(k, v)
    for i in range(0, 195, n):
        b.append(k[i:i + n], v[i:i + n])
    assert a.seq_len == b.seq_len == 195
    for name in ("k_codes", "v_codes", "k_scales", "v_scales"):
        assert torch.equal(getattr(a, name), getattr(b, name)), name
    if n <= 64:
        before = b.k_codes.clone()
        slots = np.full(n, -1, np.int32)
        slots[0] = 64 * 16                            # past the last page
        p = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())
        rc = pkg.lib().ojasx_kv_encode_append_host_slots(
            p(k), p(v), n, 2, 64, 16, p(b.k_codebook) if codebook else None,
            p(b.v_codebook) if codebook else None, slots.ctypes.data, 16, 64, p(b.k_codes),
            p(b.k_scales), p(b.v_codes), p(b.v_scales), None)
        assert rc == 0
        torch.cuda.synchronize()
        assert torch.equal(before, b.k_codes)


@pytest.mark.parametrize("n", [1, 64, 65])
def test_append_refuses_capture(pkg, dev, n):
    """A captured append would write the same slots on every replay: it raises before the page
    table moves, and the capture and later appends go on."""
    import torch
    cache = pkg.long_context.PagedCodeKVCache(2, 64, 16, page_size=16, max_resident_pages=8,
                                              sink_pages=1, device=dev)
    x = torch.randn(n, 2, 64, device=dev)
    cache.append(x[:1], x[:1])
    codes, a = cache.k_codes.clone(), torch.zeros(4, device=dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        a.add_(1)
        with pytest.raises(RuntimeError, match="captured"):
            cache.append(x, x)
    for i in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert (a == i + 1).all()
    assert cache.seq_len == cache.total_tokens_seen == 1 and torch.equal(cache.k_codes, codes)
    cache.append(x, x)
    assert cache.seq_len == cache.total_tokens_seen == 1 + n


def test_host_slots_refuses_more_than_64(pkg, dev):
    import torch
    t = torch.zeros(65, 1, 16, device=dev)
    u = torch.zeros(65 * 16, dtype=torch.uint8, device=dev)
    p = lambda a: ctypes.c_void_p(a.data_ptr())
    rc = pkg.lib().ojasx_kv_encode_append_host_slots(
        p(t), p(t), 65, 1, 16, 16, None, None, np.zeros(65, np.int32).ctypes.data, 16, 8, p(u), p(t), p(u),
        p(t), None)
    assert rc == -3
