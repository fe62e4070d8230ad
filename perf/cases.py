"""Performance cases of the LUT engine: what a program that uses it runs, through its public
entry points, over the sizes, types and options that it meets.

``listed()`` holds the named cases, ``draw(rng)`` one more case of the same ranges.  A case's
``kind`` names the entry point:

* ``linear``   ``engine.SplitManifoldLUTLinear.forward``, one token to a prefill chunk;
* ``grouped``  ``ojasx_linear_forward_grouped_device``: many one-token linears in one call;
* ``moe``      router and top-k expert layer (``ojasx_moe_route_device``,
               ``ojasx_moe_forward_device``), one token to a prefill chunk;
* ``kv``       a decode step of one attention layer on ``PagedCodeKVCache``: append the new
               token's K and V, attend over the cache;
* ``pages``    exact attention over the int8 pages of a ``PagedCompressedKVCache``: one decode
               query, or a prefill chunk that is appended first;
* ``attn``     ``OnlineSoftmaxBlockAttention.forward`` over K/V tensors;
* ``rvq``      ``math_engine.subspace_lut_rvq_gemm``, the residual-VQ linear;
* ``decoder``  ``LUTDecoder.generate``: greedy tokens of a stack of layers with its LM head.

Weights and inputs follow the distributions of the package's ``synthetic`` module.
"""
import ctypes
import math

import numpy as np
import torch

import __graft_entry__

pkg = __graft_entry__.load_package()

DENSITY, SIGMA = 0.0038, 0.02       # outliers per weight and the weights' spread
PAGE = 16                           # tokens of a code-domain KV page


def listed():
    return [
        # one token through a square projection: the smallest call a decode loop makes
        dict(name="linear_1tok", kind="linear", tokens=1, K=2560, M=2560, bf16=False, bias=False),
        # eight sequences decoding together through the gate/up projection, a bf16 model
        dict(name="linear_8tok_bf16", kind="linear", tokens=8, K=2560, M=6912, bf16=True, bias=False),
        # a large decode batch (or a short prompt) through the same projection in fp32
        dict(name="linear_64tok", kind="linear", tokens=64, K=2560, M=6912, bf16=False, bias=False),
        # a prefill chunk of a bf16 model
        dict(name="linear_2048tok_bf16", kind="linear", tokens=2048, K=2560, M=6912, bf16=True, bias=False),
        # independent one-token projections of several streams or layers in one call
        dict(name="grouped_64", kind="grouped", count=64, K=2560, M=6912),
        # the 512-expert top-10 layer on a decode batch
        dict(name="moe_16tok", kind="moe", tokens=16, E=512, H=2048, I=768, k=10, bf16=False),
        # the same layer on a prefill chunk
        dict(name="moe_1024tok", kind="moe", tokens=1024, E=512, H=2048, I=768, k=10, bf16=False),
        # a decode step at a long context, the cache at its page limit
        dict(name="kv_step_32k", kind="kv", tokens=32768, q_heads=32, kv_heads=8),
        # one decode query, exact, over a long int8 cache
        dict(name="pages_32k_1q", kind="pages", tokens=32768, q_len=1, q_heads=32, kv_heads=8, D=128, bf16=False),
        # exact attention of a prompt chunk over itself and the context before it
        dict(name="attn_prefill_512", kind="attn", tokens=2048, q_len=512, q_heads=32, kv_heads=8, D=128,
             dtype="bf16", causal=True),
        # a two-stage residual-VQ projection on a decode batch
        dict(name="rvq_32tok", kind="rvq", tokens=32, rows=6912, cols=2560, block=16, bits=8, stages=2,
             bf16=False, bias=False),
        # greedy decoding with the 4B shape's widths, LM head and context (six of its layers)
        dict(name="decoder_6layer", kind="decoder", layers=6, hidden=2560, intermediate=9728, vocab=151936,
             context=4096, new_tokens=8),
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "grouped", "moe", "moe", "kv", "pages", "attn", "rvq",
                       "rvq", "decoder"])
    if kind == "linear":
        K, M = 16 * _log(rng, 32, 608), _log(rng, 512, 19456)
        tokens = min(_log(rng, 1, 2048), 2048 * 2560 * 6912 // (K * M))
        bf16 = rng.random() < 0.5
        return dict(kind=kind, tokens=max(1, tokens if bf16 else tokens // 2), K=K, M=M, bf16=bf16,
                    bias=rng.random() < 0.3)
    if kind == "grouped":
        return dict(kind=kind, count=_log(rng, 4, 96), K=16 * _log(rng, 64, 160), M=_log(rng, 1024, 6912))
    if kind == "moe":
        E = rng.choice([64, 128, 256])
        return dict(kind=kind, tokens=_log(rng, 1, 1024), E=E, H=16 * rng.randint(64, 128),
                    I=16 * rng.randint(32, 48), k=rng.choice([4, 6, 8, 10]), bf16=rng.random() < 0.4)
    if kind == "kv":
        kvh = rng.choice([4, 8])
        return dict(kind=kind, tokens=_log(rng, 100, 32768), q_heads=4 * kvh, kv_heads=kvh)
    if kind == "pages":
        q_len = rng.choice([1, 1, 64, 128, 256])
        return dict(kind=kind, tokens=_log(rng, 600, 32768 if q_len == 1 else 4096), q_len=q_len,
                    q_heads=rng.choice([16, 32]), kv_heads=rng.choice([4, 8]), D=rng.choice([64, 128, 128]),
                    bf16=rng.random() < 0.5)
    if kind == "attn":
        q_len = _log(rng, 1, 768)
        return dict(kind=kind, tokens=q_len + rng.randint(0, 1400), q_len=q_len, q_heads=rng.choice([16, 32]),
                    kv_heads=rng.choice([2, 4, 8, 16]), D=rng.choice([64, 80, 128, 128]),
                    dtype=rng.choice(["f32", "bf16", "bf16", "f16"]), causal=rng.random() < 0.8)
    if kind == "rvq":
        block, bits = rng.choice([(16, 8), (16, 8), (8, 8), (8, 4), (16, 4), (4, 4), (24, 2), (32, 8)])
        return dict(kind=kind, tokens=_log(rng, 1, 128), rows=_log(rng, 256, 6912), cols=_log(rng, 256, 2560),
                    block=block, bits=bits, stages=rng.choice([1, 2, 2, 3]), bf16=rng.random() < 0.5,
                    bias=rng.random() < 0.5)
    return dict(kind=kind, layers=rng.randint(1, 3), hidden=128 * rng.randint(8, 20),
                intermediate=128 * rng.randint(24, 76), vocab=_log(rng, 16384, 151936),
                context=_log(rng, 64, 4096), new_tokens=rng.randint(1, 8))


def work(case):
    c = case
    if c["kind"] == "linear":
        B, K, M = c["tokens"], c["K"], c["M"]
        e = 2 if c["bf16"] else 4
        return dict(bytes=_linear_bytes(K, M) + e * B * (K + M), flops=2 * B * K * M)
    if c["kind"] == "grouped":
        K, M = c["K"], c["M"]
        return dict(bytes=c["count"] * (_linear_bytes(K, M) + 4 * (K + M)), flops=2 * c["count"] * K * M)
    if c["kind"] == "moe":
        T, E, H, I, k = c["tokens"], c["E"], c["H"], c["I"], c["k"]
        e = 2 if c["bf16"] else 4
        distinct = E * (1 - (1 - k / E) ** T)           # experts a batch of T tokens routes to
        expert = 2 * I * (H // 16) + H * (I // 16) + 4 * (2 * I + H)
        return dict(bytes=distinct * expert + T * (2 * e * H + 4 * E), flops=6 * T * k * H * I)
    if c["kind"] == "kv":
        T, hk = c["tokens"], c["kv_heads"]
        return dict(bytes=T * hk * 2 * (8 + 4) + 2 * hk * 256 * 16 * 4, flops=4 * T * c["q_heads"] * 128)
    if c["kind"] in ("pages", "attn"):
        T, S, D, Hq, hk = c["tokens"], c["q_len"], c["D"], c["q_heads"], c["kv_heads"]
        e = 1 if c["kind"] == "pages" else 4 if c["dtype"] == "f32" else 2
        causal = c["kind"] == "pages" or c["causal"]
        pairs = S * T - S * (S - 1) // 2 if causal else S * T
        return dict(bytes=2 * T * hk * D * e + 2 * 2 * S * Hq * D, flops=4 * pairs * Hq * D)
    if c["kind"] == "rvq":
        B, R, K = c["tokens"], c["rows"], c["cols"]
        e = 2 if c["bf16"] else 4
        G = -(-K // c["block"])
        return dict(bytes=c["stages"] * R * G * c["bits"] // 8 + 4 * R + e * B * (K + R), flops=2 * B * R * K)
    h, i, n = c["hidden"], c["intermediate"], c["layers"]
    shapes = n * [(h, 6144), (4096, h), (h, 2 * i), (i, h)] + [(h, c["vocab"])]
    weights = sum(_linear_bytes(K, M) for K, M in shapes) + n * c["context"] * 8 * 2 * (8 + 4)
    macs = sum(K * M for K, M in shapes) + n * c["context"] * 32 * 128 * 2
    return dict(bytes=c["new_tokens"] * weights, flops=c["new_tokens"] * 2 * macs)


def _linear_bytes(K, M):
    """Codes, scales and outliers (16-bit column, fp32 value) of one LUT linear."""
    return M * (K // 16) + 4 * M + 4 * (M + 1) + 6 * int(DENSITY * K * M)


def tolerance(case):
    c = case
    if c.get("bf16") or c.get("dtype") == "bf16":
        return {"rel": 4e-3, "max": 5e-2}       # the outputs' own rounding: 1.7e-3 from exact()
    if c.get("dtype") == "f16":
        return {"rel": 1e-3, "max": 2e-2}       # the same at 11 bits
    if c["kind"] == "decoder":
        return {"rel": 5e-6, "max": 1e-3}       # fp32 through all layers: 5.4e-7 from exact()
    return {"rel": 2e-6, "max": 1e-4}           # fp32 sums: 0.6e-7 .. 3.1e-7 from exact()


# ---- inputs, on the GPU, from the seed alone ------------------------------------------------


def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _uniform(g, lo, hi, *shape):
    return torch.rand(*shape, generator=g, device="cuda") * (hi - lo) + lo


def _codes(g, *shape, n=256):
    return torch.randint(0, n, shape, generator=g, device="cuda", dtype=torch.uint8)


def _outliers(g, M, K):
    """Sorted distinct positions (row * K + column) and values of the exact weights."""
    pos = torch.randint(0, M * K, (int(DENSITY * M * K),), generator=g, device="cuda").unique()
    mag = _uniform(g, 15 * SIGMA, 36 * SIGMA, pos.numel())
    return pos, torch.where(torch.rand(pos.numel(), generator=g, device="cuda") < 0.5, -mag, mag)


def _csr(pos, M, K):
    rows = torch.zeros(M + 1, dtype=torch.int64, device="cuda")
    rows[1:] = torch.bincount(pos // K, minlength=M).cumsum(0)
    return rows.int().cpu().numpy(), (pos % K).int().cpu().numpy()


def _linear_weights(g, M, K, unit_scales=False):
    cb, codes = _normal(g, 256, 16, std=SIGMA), _codes(g, M, K // 16)
    scales = torch.ones(M, device="cuda") if unit_scales else _uniform(g, 0.5, 1.5, M)
    return dict(cb=cb, codes=codes, scales=scales, out=_outliers(g, M, K))


def _dense(w, K):
    """A LUT linear's weight matrix in 64 bits."""
    W = w["cb"].double()[w["codes"].long()].flatten(1) * w["scales"].double()[:, None]
    W.view(-1)[w["out"][0]] += w["out"][1].double()
    return W


def _native(w, M, K):
    lin = pkg.native.NativeSplitManifoldLinear(K, M, 16, 256)
    lin.initialize_weights(w["cb"].cpu().numpy(), w["codes"].cpu().numpy(), w["scales"].cpu().numpy())
    rp, cl = _csr(w["out"][0], M, K)
    lin.set_outliers(rp, cl, w["out"][1].cpu().numpy())
    return lin


def _vp(t):
    return ctypes.c_void_p(t.data_ptr())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


# ---- linear ----------------------------------------------------------------------------------


def _linear_inputs(c, seed):
    g, dt = _gen(seed), torch.bfloat16 if c["bf16"] else torch.float32
    w = _linear_weights(g, c["M"], c["K"])
    w = {k: v.to(dt) if k in ("cb", "scales") else v for k, v in w.items()}
    w["out"] = (w["out"][0], w["out"][1].to(dt))
    bias = _normal(g, c["M"], std=0.1).to(dt) if c["bias"] else None
    return w, bias, _normal(g, c["tokens"], c["K"]).to(dt), dt


def _linear_prepare(c, seed):
    w, bias, x, dt = _linear_inputs(c, seed)
    layer = pkg.engine.SplitManifoldLUTLinear(c["K"], c["M"], bias=c["bias"], dtype=dt).to("cuda")
    layer.codebook.copy_(w["cb"])
    layer.codes.copy_(w["codes"])
    layer.scales.copy_(w["scales"])
    pos, val = w["out"]
    layer.outlier_indices = torch.stack([pos // c["K"], pos % c["K"]])
    layer.outlier_values = val
    layer.num_outliers = val.numel()
    if bias is not None:
        layer.bias.data.copy_(bias)
    with torch.no_grad():
        layer(torch.zeros_like(x[:1]))          # lays the weights out, as a loaded model has them
    return dict(layer=layer, x=x)


def _linear_run(s):
    with torch.no_grad():
        return s["layer"](s["x"])


def _linear_exact(c, seed):
    w, bias, x, _ = _linear_inputs(c, seed)
    y = x.double() @ _dense(w, c["K"]).t()
    return y if bias is None else y + bias.double()


# ---- grouped linears -------------------------------------------------------------------------


def _grouped_inputs(c, seed):
    g = _gen(seed)
    return [(_linear_weights(g, c["M"], c["K"], unit_scales=True), _normal(g, c["K"])) for _ in range(c["count"])]


def _grouped_prepare(c, seed):
    items = _grouped_inputs(c, seed)
    lins = [_native(w, c["M"], c["K"]) for w, _ in items]
    xs, y = [x for _, x in items], torch.empty(c["count"], c["M"], device="cuda")
    ptrs = lambda v: (ctypes.c_void_p * len(v))(*v)
    return dict(lins=lins, xs=xs, y=y, n=c["count"], handles=ptrs([lin.handle for lin in lins]),
                xp=ptrs([x.data_ptr() for x in xs]), yp=ptrs([r.data_ptr() for r in y]))


def _grouped_run(s):
    pkg._lib.check(pkg._lib.lib().ojasx_linear_forward_grouped_device(
        s["handles"], s["n"], s["xp"], s["yp"], _stream()), "grouped")
    return s["y"]


def _grouped_exact(c, seed):
    return torch.stack([_dense(w, c["K"]) @ x.double() for w, x in _grouped_inputs(c, seed)])


# ---- mixture of experts ----------------------------------------------------------------------


def _moe_inputs(c, seed):
    g, E, H, I = _gen(seed), c["E"], c["H"], c["I"]
    return dict(cb_in=_normal(g, 256, 16, std=SIGMA), cb_dn=_normal(g, 256, 16, std=SIGMA),
                gu=_codes(g, E, 2 * I, H // 16), dn=_codes(g, E, H, I // 16),
                gs=_uniform(g, 0.5, 1.5, E, 2 * I), ds=_uniform(g, 0.5, 1.5, E, H),
                x=_normal(g, c["tokens"], H).to(torch.bfloat16 if c["bf16"] else torch.float32),
                logits=_normal(g, c["tokens"], E))


def _moe_prepare(c, seed):
    m = _moe_inputs(c, seed)
    layer = pkg.native.NativeSplitManifoldMoE(c["E"], c["H"], c["I"], c["k"], 16)
    layer.initialize_weights(*[m[k].cpu().numpy() for k in ("cb_in", "cb_dn", "gu", "gs", "dn", "ds")])
    T, k = c["tokens"], c["k"]
    return dict(layer=layer, x=m["x"], logits=m["logits"], T=T, E=c["E"], k=k, tag=1 if c["bf16"] else 0,
                idx=torch.empty(T, k, dtype=torch.int32, device="cuda"), w=torch.empty(T, k, device="cuda"),
                y=torch.empty_like(m["x"]))


def _moe_run(s):
    L, st = pkg._lib.lib(), _stream()
    pkg._lib.check(L.ojasx_moe_route_device(_vp(s["logits"]), s["T"], s["E"], s["k"], 1, _vp(s["idx"]),
                                            _vp(s["w"]), st), "route")
    pkg._lib.check(L.ojasx_moe_forward_device(s["layer"].handle, _vp(s["x"]), _vp(s["idx"]), _vp(s["w"]),
                                              _vp(s["y"]), s["T"], s["k"], s["tag"], st), "moe")
    return dict(y=s["y"], idx=s["idx"], w=s["w"])


def _moe_exact(c, seed):
    m = _moe_inputs(c, seed)
    top, idx = torch.topk(m["logits"].double(), c["k"])
    w = torch.softmax(top, dim=1)
    x, y = m["x"].double(), torch.zeros(c["tokens"], c["H"], dtype=torch.float64, device="cuda")
    cin, cdn, I = m["cb_in"].double(), m["cb_dn"].double(), c["I"]
    for e in idx.unique().tolist():
        t, slot = (idx == e).nonzero(as_tuple=True)
        z = x[t] @ cin[m["gu"][e].long()].flatten(1).t() * m["gs"][e].double()
        a = torch.nn.functional.silu(z[:, :I]) * z[:, I:]
        y.index_add_(0, t, w[t, slot, None] * (a @ cdn[m["dn"][e].long()].flatten(1).t() * m["ds"][e].double()))
    return dict(y=y, idx=None, w=w)


# ---- code-domain KV cache --------------------------------------------------------------------


def _kv_inputs(c, seed):
    g, T, h = _gen(seed), c["tokens"], c["kv_heads"]
    return dict(kcb=_normal(g, h, 256, 16, std=40.0), vcb=_normal(g, h, 256, 16, std=40.0),
                k=_normal(g, T, h, 128), v=_normal(g, T, h, 128), kn=_normal(g, 1, h, 128),
                vn=_normal(g, 1, h, 128), q=_normal(g, c["q_heads"], 128))


def _kv_pages(c):
    return max(4, -(-c["tokens"] // PAGE))


def _kv_prepare(c, seed):
    m = _kv_inputs(c, seed)
    cache = pkg.long_context.PagedCodeKVCache(c["kv_heads"], 128, 16, page_size=PAGE,
                                              max_resident_pages=_kv_pages(c), sink_pages=2,
                                              k_codebook=m["kcb"], v_codebook=m["vcb"])
    cache.append(m["k"], m["v"])
    return dict(cache=cache, kn=m["kn"], vn=m["vn"], q=m["q"])


def _kv_run(s):
    cache = s["cache"]
    cache.append(s["kn"], s["vn"])
    out = cache.decode(s["q"])
    return dict(out=out, k_codes=cache.k_codes, v_codes=cache.v_codes, k_scales=cache.k_scales,
                v_scales=cache.v_scales)


def _kv_encode(x, cb):
    """x [T, 128] through the cache's encoder, which is defined in fp32: the values its codes
    and scale stand for, in 64 bits."""
    s = x.abs().amax(1, keepdim=True).clamp(min=1e-8)
    s = s / torch.full_like(s, 127.0)
    n, best = x / s, []
    for g in range(8):
        d2 = torch.zeros(x.shape[0], 256, device="cuda")
        for d in range(16):
            diff = (n[:, 16 * g + d, None] - cb[None, :, d]).double()
            d2 = (d2.double() + diff * diff).float()
        best.append(d2.argmin(1))
    return (cb.double()[torch.stack(best, 1)] * s.double()[:, :, None]).flatten(1)


def _kv_exact(c, seed):
    m = _kv_inputs(c, seed)
    T, cap, R = c["tokens"], PAGE * _kv_pages(c), c["q_heads"] // c["kv_heads"]
    keep = torch.arange(T, device="cuda")
    if T == cap:                                # the new token's page takes the oldest one's place
        keep = torch.cat([keep[:2 * PAGE], keep[3 * PAGE:]])
    out = []
    for h in range(c["kv_heads"]):
        K = _kv_encode(torch.cat([m["k"][keep, h], m["kn"][:, h]]), m["kcb"][h])
        V = _kv_encode(torch.cat([m["v"][keep, h], m["vn"][:, h]]), m["vcb"][h])
        p = torch.softmax(m["q"][R * h:R * h + R].double() @ K.t() / math.sqrt(128), 1)
        out.append(p @ V)
    return dict(out=torch.cat(out), k_codes=None, v_codes=None, k_scales=None, v_scales=None)


# ---- exact attention over int8 pages ---------------------------------------------------------


def _pages_inputs(c, seed):
    g, dt = _gen(seed), torch.bfloat16 if c["bf16"] else torch.float32
    h, D, T, S = c["kv_heads"], c["D"], c["tokens"], c["q_len"]
    return dict(k=_normal(g, 1, h, T, D).to(dt), v=_normal(g, 1, h, T, D).to(dt),
                kn=_normal(g, 1, h, S, D).to(dt), vn=_normal(g, 1, h, S, D).to(dt),
                q=_normal(g, 1, c["q_heads"], S, D).to(dt))


def _pages_size(c):
    """Tokens of a page: a prefill chunk fills one; decode queries read pages of 256."""
    return 256 if c["q_len"] == 1 else c["q_len"]


def _pages_prepare(c, seed):
    m, page = _pages_inputs(c, seed), _pages_size(c)
    cache = pkg.long_context.PagedCompressedKVCache(page, max_resident_pages=max(4, -(-c["tokens"] // page)),
                                                    sink_pages=2)
    cache.append(m["k"], m["v"])
    att = pkg.long_context.OnlineSoftmaxBlockAttention(c["q_heads"], c["kv_heads"], c["D"], causal=True)
    return dict(cache=cache, att=att, q=m["q"], kn=m["kn"], vn=m["vn"])


def _pages_run(s):
    cache, S = s["cache"], s["q"].shape[2]
    page = None
    if S > 1:                                   # a prefill chunk: its keys are attended to as well
        cache.append(s["kn"], s["vn"])
        page = cache._pages[-1]
    out, report = s["att"].forward_stream(s["q"], cache, query_start_pos=cache.resident_tokens - S)
    return dict(out=out, lse=report.max_logsumexp, page=page)


def _page_values(t):
    """[.., D] through the int8 pages' quantiser (per-token scale, in t's type, stored in fp16)."""
    s = t.abs().amax(-1, keepdim=True).clamp(min=1e-8)
    s = s / torch.full_like(s, 127.0)
    q = torch.round(t / s).clamp(-127, 127)
    return q.double() * s.half().double()


def _pages_exact(c, seed):
    m, page, T, S = _pages_inputs(c, seed), _pages_size(c), c["tokens"], c["q_len"]
    k, v = m["k"], m["v"]
    if S > 1:
        keep = torch.arange(T, device="cuda")
        if -(-T // page) >= 4:                  # full: the oldest page after the first two goes
            keep = torch.cat([keep[:2 * page], keep[3 * page:]])
        k, v = torch.cat([k[:, :, keep], m["kn"]], 2), torch.cat([v[:, :, keep], m["vn"]], 2)
    out, lse = _attention(m["q"], _page_values(k), _page_values(v), True, k.shape[2] - S)
    return dict(out=out, lse=lse, page=None if S == 1 else [None] * 4)


def _attention(q, k, v, causal, start):
    """softmax(q k^T / sqrt(D)) v in 64 bits and the largest log-sum-exp of a row."""
    B, Hq, S, D = q.shape
    R, T = Hq // k.shape[1], k.shape[2]
    out, lse = torch.empty(B, Hq, S, D, dtype=torch.float64, device="cuda"), -math.inf
    for h in range(Hq):
        s = q[0, h].double() @ k[0, h // R].double().t() / math.sqrt(D)
        if causal:
            hide = torch.arange(T, device="cuda")[None, :] > start + torch.arange(S, device="cuda")[:, None]
            s = s.masked_fill(hide, -math.inf)
        out[0, h] = torch.softmax(s, 1) @ v[0, h // R].double()
        lse = max(lse, float(torch.logsumexp(s, 1).max()))
    return out, lse


# ---- exact attention over tensors ------------------------------------------------------------


def _attn_inputs(c, seed):
    g, dt = _gen(seed), {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[c["dtype"]]
    h, D, T, S = c["kv_heads"], c["D"], c["tokens"], c["q_len"]
    return (_normal(g, 1, c["q_heads"], S, D).to(dt), _normal(g, 1, h, T, D).to(dt),
            _normal(g, 1, h, T, D).to(dt))


def _attn_prepare(c, seed):
    q, k, v = _attn_inputs(c, seed)
    att = pkg.long_context.OnlineSoftmaxBlockAttention(c["q_heads"], c["kv_heads"], c["D"], causal=c["causal"])
    return dict(att=att, q=q, k=k, v=v, start=c["tokens"] - c["q_len"])


def _attn_run(s):
    return s["att"].forward(s["q"], s["k"], s["v"], query_start_pos=s["start"])


def _attn_exact(c, seed):
    q, k, v = _attn_inputs(c, seed)
    return _attention(q, k, v, c["causal"], c["tokens"] - c["q_len"])[0]


# ---- residual-VQ linear ----------------------------------------------------------------------


def _rvq_inputs(c, seed):
    g, dt = _gen(seed), torch.bfloat16 if c["bf16"] else torch.float32
    S, R, G, Q = c["stages"], c["rows"], -(-c["cols"] // c["block"]), 1 << c["bits"]
    # each stage codes what the one before left: about half its size
    cbs = torch.stack([_normal(g, Q, c["block"], std=SIGMA * 0.5 ** s) for s in range(S)])
    return dict(cbs=cbs, codes=_codes(g, S, R * G, n=Q), scales=_uniform(g, 0.5, 1.5, R),
                bias=_normal(g, R, std=0.1) if c["bias"] else None, x=_normal(g, c["tokens"], c["cols"]).to(dt))


def _rvq_prepare(c, seed):
    m, per = _rvq_inputs(c, seed), 8 // c["bits"]
    codes = torch.nn.functional.pad(m["codes"], (0, -m["codes"].shape[1] % per)).view(c["stages"], -1, per)
    packed = torch.zeros(codes.shape[:2], dtype=torch.uint8, device="cuda")
    for i in range(per):
        packed |= codes[:, :, i] << (i * c["bits"])
    enc = pkg.math_engine.QuantizedWeight((c["rows"], c["cols"]), c["block"], c["bits"], packed, m["cbs"],
                                          m["scales"])
    return dict(enc=enc, x=m["x"], bias=m["bias"])


def _rvq_run(s):
    return pkg.math_engine.subspace_lut_rvq_gemm(s["x"], s["enc"], s["bias"])


def _rvq_exact(c, seed):
    m = _rvq_inputs(c, seed)
    W = sum(m["cbs"][s].double()[m["codes"][s].long()] for s in range(c["stages"]))
    W = W.reshape(c["rows"], -1)[:, :c["cols"]] * m["scales"].double()[:, None]
    y = m["x"].double() @ W.t()
    return y if m["bias"] is None else y + m["bias"].double()


# ---- decoder ---------------------------------------------------------------------------------

_Q, _KV, _EPS, _THETA = 32, 8, 1e-6, 1e6


def _decoder_inputs(c, seed):
    g, h, i = _gen(seed), c["hidden"], c["intermediate"]
    pages = -(-c["context"] // PAGE)
    lin = lambda M, K: _linear_weights(g, M, K, unit_scales=True)
    layers = []
    for _ in range(c["layers"]):
        layers.append(dict(
            qkv=lin((_Q + 2 * _KV) * 128, h), o=lin(h, _Q * 128), gate_up=lin(2 * i, h), down=lin(h, i),
            norms=[_uniform(g, 0.8, 1.2, n) for n in (h, h, 128, 128)],
            kcb=_normal(g, _KV, 256, 16, std=40.0), vcb=_normal(g, _KV, 256, 16, std=40.0),
            kc=_codes(g, pages, _KV, PAGE, 8), vc=_codes(g, pages, _KV, PAGE, 8),
            ks=_uniform(g, 0.5, 1.5, pages, _KV, PAGE) * 3 / 127, vs=_uniform(g, 0.5, 1.5, pages, _KV, PAGE) * 3 / 127))
    return dict(layers=layers, head=lin(c["vocab"], h), norm=_uniform(g, 0.8, 1.2, h),
                emb=_normal(g, c["vocab"], h), first=int(seed) % c["vocab"])


def _decoder_prepare(c, seed):
    m, h, i = _decoder_inputs(c, seed), c["hidden"], c["intermediate"]
    D = pkg.decoder
    cfg = D.DecoderConfig(hidden=h, layers=c["layers"], q_heads=_Q, kv_heads=_KV, head_dim=128, intermediate=i,
                          vocab=c["vocab"], max_context=c["context"] + 128, page_size=PAGE, max_steps=128,
                          rms_eps=_EPS, rope_theta=_THETA)
    dec = D.LUTDecoder(cfg)
    shapes = dict(qkv=((_Q + 2 * _KV) * 128, h), o=(h, _Q * 128), gate_up=(2 * i, h), down=(h, i))
    for n, w in enumerate(m["layers"]):
        dec.set_layer(n, *[_native(w[k], *shapes[k]) for k in ("qkv", "o", "gate_up", "down")], *w["norms"],
                      w["kcb"], w["vcb"])
        dec.set_context(n, w["kc"], w["ks"], w["vc"], w["vs"], c["context"])
    dec.set_head(_native(m["head"], c["vocab"], h), m["norm"], m["emb"])
    return dict(dec=dec, first=m["first"], context=c["context"], n=c["new_tokens"])


def _decoder_run(s):
    s["dec"].reset(s["context"])
    tokens, logits = s["dec"].generate(s["first"], s["n"], return_logits=True)
    return dict(tokens=tokens, logits=logits)


def _decoder_exact(c, seed):
    m, ctx, hd = _decoder_inputs(c, seed), c["context"], 128
    rms = lambda x, w: x / torch.sqrt((x * x).mean(-1, keepdim=True) + _EPS) * w.double()
    # the rotation's angles are fp32 by definition: position times the frequency, both fp32
    freq = (1.0 / np.power(np.float64(_THETA), np.arange(64) * 2 / hd)).astype(np.float32)

    def rope(x, pos):
        a = torch.from_numpy((np.float32(pos) * freq).astype(np.float64)).cuda()
        co, si = a.cos().float().double(), a.sin().float().double()
        return torch.cat([x[:, :64] * co - x[:, 64:] * si, x[:, 64:] * co + x[:, :64] * si], 1)

    def cached(codes, scales, cb):
        k = cb.double()[torch.arange(_KV, device="cuda")[None, :, None, None], codes.long()].flatten(3)
        k = k * scales.double()[..., None]
        return [k[:, h].reshape(-1, hd)[:ctx] for h in range(_KV)]

    layers = []
    for w in m["layers"]:
        W = {k: _dense(w[k], w[k]["codes"].shape[1] * 16) for k in ("qkv", "o", "gate_up", "down")}
        layers.append((w, W, cached(w["kc"], w["ks"], w["kcb"]), cached(w["vc"], w["vs"], w["vcb"])))
    head, token = _dense(m["head"], c["hidden"]), m["first"]
    for step in range(c["new_tokens"]):
        x = m["emb"][token].double()
        for w, W, K, V in layers:
            z = (W["qkv"] @ rms(x, w["norms"][0])).view(-1, hd)
            q = rope(rms(z[:_Q], w["norms"][2]), ctx + step)
            k, v = rope(rms(z[_Q:_Q + _KV], w["norms"][3]), ctx + step), z[_Q + _KV:]
            att = []
            for h in range(_KV):
                K[h] = torch.cat([K[h], _kv_encode(k[h:h + 1].float(), w["kcb"][h])])
                V[h] = torch.cat([V[h], _kv_encode(v[h:h + 1].float(), w["vcb"][h])])
                att.append(torch.softmax(q[4 * h:4 * h + 4] @ K[h].t() / math.sqrt(hd), 1) @ V[h])
            x = x + W["o"] @ torch.cat(att).flatten()
            z = W["gate_up"] @ rms(x, w["norms"][1])
            i = z.numel() // 2
            x = x + W["down"] @ (torch.nn.functional.silu(z[:i]) * z[i:])
        logits = head @ rms(x, m["norm"])
        token = int(logits.argmax())
    return dict(tokens=None, logits=logits)


# ---- the interface ---------------------------------------------------------------------------

_KINDS = {
    "linear": (_linear_prepare, _linear_run, _linear_exact),
    "grouped": (_grouped_prepare, _grouped_run, _grouped_exact),
    "moe": (_moe_prepare, _moe_run, _moe_exact),
    "kv": (_kv_prepare, _kv_run, _kv_exact),
    "pages": (_pages_prepare, _pages_run, _pages_exact),
    "attn": (_attn_prepare, _attn_run, _attn_exact),
    "rvq": (_rvq_prepare, _rvq_run, _rvq_exact),
    "decoder": (_decoder_prepare, _decoder_run, _decoder_exact),
}


def prepare(case, seed):
    return dict(kind=case["kind"], state=_KINDS[case["kind"]][0](case, seed))


def run(state):
    return _KINDS[state["kind"]][1](state["state"])


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)
