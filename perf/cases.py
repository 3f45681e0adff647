"""The work a user of this library has it do, as cases that can be timed.

Seven kinds of call, each through the entry point a program uses:

  gemv     one weight-quantized linear layer of a decode step (Lib.gemv)
  gemm     quantize the activations per token, then the INT8 / FP8 matrix
           product of a prefill (Lib.quant_rows_*, Lib.gemm)
  proj     fp32 activations against two weight matrices that share them, the
           gate / up projections of a prefill pass (Lib.gemm_f32_multi)
  attn     LSH route + sparse attention of one decode token per sequence over
           its paged KV cache (Lib.lsh_attention)
  sample   the next token from the logits (Lib.sample_top_p / _temperature)
  step     a whole decode step (Decoder.step): logits and the K/V page written
  prefill  a whole prompt (KVPool.reset, Decoder.prefill): logits and the cache

Shapes are those of the benchmark's workloads (bench.py): the tiny decoder
(TINY), the 3B-class decoder (B3), the GEMV shapes and the 32-head attention.

`exact` restates each call in 64 bits with plain torch.  The exponential of
the attention and of SiLU is part of the path's definition (Schraudolph's
exponential: a linear map onto the bits of a float), as are the storage
formats of weights and cache, the order in which the pages are visited and the
hashing that selects them, so those are restated too.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "42-berlin-engine_amd"))
import be42  # noqa: E402

ARCH = {
    "tiny": dict(n_layers=4, dim=512, n_heads=8, n_kv_heads=8, head_dim=64, hidden_dim=1408, vocab=4096),
    "3b": dict(n_layers=28, dim=3072, n_heads=24, n_kv_heads=8, head_dim=128, hidden_dim=8192, vocab=128256),
}
PAGE = 16
K_SEL = 64        # pages attended per query once there are more
CAP = 64          # candidate pages the router looks at
PLANTED = 0.05    # share of the pages whose keys resemble the query
EPS, THETA = 1e-5, 1e4
F64 = torch.float64


def listed():
    return [
        # the smallest linear layer (q projection of the tiny decoder): latency and launches
        dict(name="gemv_smallest", op="gemv", kind="int8", n=512, k=512, batch=1),
        # an FFN matrix at a small serving batch
        dict(name="gemv_ffn", op="gemv", kind="int8", n=14336, k=4096, batch=4),
        # the vocabulary projection at a full batch: the largest weight of a step
        dict(name="gemv_head", op="gemv", kind="fp8", n=128256, k=4096, batch=16),
        # a short prompt, not a multiple of any tile
        dict(name="gemm_ragged", op="gemm", kind="int8", m=500, n=4096, k=4096),
        # a long prompt against an FFN matrix
        dict(name="gemm_large", op="gemm", kind="fp8", m=8192, n=14336, k=4096),
        # one user's token at a long context: latency
        dict(name="attn_one", op="attn", kv="bf16", ctx=32768, batch=1, heads=32, kv_heads=8, head_dim=128),
        # a serving batch at the same context: bandwidth
        dict(name="attn_batch", op="attn", kv="bf16", ctx=32768, batch=64, heads=32, kv_heads=8, head_dim=128),
        # nucleus sampling over a large vocabulary for a small batch
        dict(name="sample_top_p", op="sample", method="top_p", vocab=128256, batch=8, bf16=False),
        # greedy decoding of the tiny decoder: launch and barrier latency
        dict(name="step_tiny", op="step", arch="tiny", kind="int8", kv="int8", batch=1, ctx=160),
        # one user's decode step of the 3B decoder over a 32k prefix
        dict(name="step_3b_one", op="step", arch="3b", kind="fp8", kv="bf16", batch=1, ctx=32768),
        # eight users' decode step of the 3B decoder
        dict(name="step_3b_batch", op="step", arch="3b", kind="fp8", kv="bf16", batch=8, ctx=8190),
        # a prompt of the 3B decoder
        dict(name="prefill_3b", op="prefill", arch="3b", kind="fp8", kv="bf16", n=1000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gemv", "gemv", "gemm", "proj", "attn", "attn", "sample", "step", "step", "prefill"])
    kind = rng.choice(["int8", "fp8"])
    kv = rng.choice(["bf16", "bf16", "int8"])
    if op == "gemv":
        k = 16 * _log(rng, 32, 896)
        return dict(op=op, kind=kind, n=_log(rng, 512, min(128256, 128256 * 4096 // k)), k=k,
                    batch=rng.choice([1, 1, 2, 3, 4, 5, 8, 11, 16]))
    if op == "gemm":
        k, n = 16 * _log(rng, 32, 896), _log(rng, 512, 14336)
        return dict(op=op, kind=kind, m=_log(rng, 17, min(8192, 8192 * 14336 * 4096 // (n * k))), n=n, k=k)
    if op == "proj":
        return dict(op=op, kind=kind, m=_log(rng, 17, 1024), n=_log(rng, 512, 8192), k=16 * _log(rng, 32, 512))
    if op == "attn":
        heads, kv_heads, hd = rng.choice([(32, 8, 128), (24, 8, 128), (8, 8, 64)])
        ctx = _log(rng, 300, 131072)
        return dict(op=op, kv=kv, ctx=ctx, batch=_log(rng, 1, min(128, 64 * 32768 // ctx)), heads=heads,
                    kv_heads=kv_heads, head_dim=hd)
    if op == "sample":
        return dict(op=op, method=rng.choice(["top_p", "temperature"]), vocab=_log(rng, 4096, 128256),
                    batch=_log(rng, 1, 16), bf16=rng.random() < 0.3)
    arch = rng.choice(["tiny", "3b"])
    if op == "step":
        ctx = _log(rng, 30, 4000 if arch == "tiny" else 32768)
        return dict(op=op, arch=arch, kind=kind, kv=kv, batch=min(rng.choice([1, 1, 2, 3, 5, 8]), max(1, 65536 // ctx)),
                    ctx=ctx)
    return dict(op=op, arch=arch, kind=kind, kv=kv, n=_log(rng, 20, 2000 if arch == "tiny" else 1000))


# ---- inputs ------------------------------------------------------------------


def _gen(seed, *more):
    g = torch.Generator(device="cuda")
    g.manual_seed(hash((int(seed),) + more) & 0x7FFFFFFFFFFF)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _weight(g, n, k, kind):
    """N(0, 0.02) weights [n][k] as a checkpoint holds them: INT8 or E4M3
    codes with one scale per row."""
    w = _randn(g, n, k) * 0.02
    amax = w.abs().amax(1)
    if kind == "int8":
        s = amax / 127.0
        return torch.round(w / s[:, None]).clamp_(-127, 127).to(torch.int8), s
    s = amax / 224.0
    return (w / s[:, None]).to(torch.float8_e4m3fn).view(torch.uint8), s


def _dense(w, s, kind):
    """The weights a pair of codes and scales stands for, in 64 bits."""
    v = w if kind == "int8" else w.view(torch.float8_e4m3fn)
    return v.to(torch.float32).to(F64) * s.to(F64)[:, None]


def _activations(g, m, k):
    """N(0, 1) with 1% outliers at +-8."""
    x = _randn(g, m, k)
    r = torch.rand(m, k, generator=g, device="cuda")
    return torch.where(r < 0.005, -8.0, torch.where(r < 0.01, 8.0, x)).contiguous()


def _projection(hd):
    """The 16 hash directions [hd][16] (unit N(0, 1) vectors)."""
    p = np.random.default_rng(42).standard_normal((16, hd)).astype(np.float32)
    return np.ascontiguousarray((p / np.linalg.norm(p, axis=1, keepdims=True)).astype(np.float32).T)


def _history(seed, slot, ctx, kv_heads, hd, q=None):
    """A slot's prefix: N(0, 1) keys and values [ctx][kv_heads * hd].  With q
    ([heads][hd]), 5% of the pages (not the first or last) have keys along the
    mean query on every head, as tokens relevant to it would."""
    g = _gen(seed, slot)
    k, v = _randn(g, ctx, kv_heads * hd), _randn(g, ctx, kv_heads * hd)
    pages = ctx // PAGE
    n = int(round(PLANTED * pages))
    if q is not None and n and pages > 2:
        u = q.to(F64).mean(0)
        u = (6.0 * u / u.norm()).to(torch.float32)
        at = torch.randperm(pages - 2, generator=g, device="cuda")[:n] + 1
        rows = (at[:, None] * PAGE + torch.arange(PAGE, device="cuda")).reshape(-1)
        k.view(ctx, kv_heads, hd)[rows] = u + 0.05 * _randn(g, rows.numel(), kv_heads, hd)
    return k, v


def _model(case, seed):
    """Weights of a decoder of the case's architecture."""
    a, g, kind = ARCH[case["arch"]], _gen(seed), case["kind"]
    d, f = a["dim"], a["hidden_dim"]
    qd, kd = a["n_heads"] * a["head_dim"], a["n_kv_heads"] * a["head_dim"]

    def norm():
        return (1.0 + 0.1 * _randn(g, d)).to(torch.bfloat16)

    layers = []
    for _ in range(a["n_layers"]):
        one = {}
        for name, (n, k) in dict(q=(qd, d), k=(kd, d), v=(kd, d), o=(d, qd), **{"1": (f, d), "3": (f, d), "2": (d, f)}).items():
            one["w" + name], one["s" + name] = _weight(g, n, k, kind)
        one["attn_norm"], one["ffn_norm"] = norm(), norm()
        layers.append(one)
    emb, emb_s = _weight(g, a["vocab"], d, kind)
    out, out_s = _weight(g, a["vocab"], d, kind)
    return dict(layers=layers, emb=emb, emb_s=emb_s, out=out, out_s=out_s, final_norm=norm())


def _tokens(case, seed, n):
    return np.random.default_rng(seed).integers(0, ARCH[case["arch"]]["vocab"], n).astype(np.int32)


def _kv_kind(name):
    return be42.KV_BF16 if name == "bf16" else be42.KV_INT8


class _Array:
    """A device array of a decoder's page pool, for torch.as_tensor, whose
    tensors keep this object, and with it the decoder and its memory."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr=typestr, version=2, strides=None)


def _pool_views(dec):
    """K and V of every page of the decoder's pool as torch tensors on its own memory."""
    s = dec.pool.s
    pages, heads, hd = s.capacity, s.n_kv, s.head_dim
    if s.kind == be42.KV_BF16:
        k = torch.as_tensor(_Array(dec, s.k, (pages, heads, PAGE, hd), "<i2"), device="cuda").view(torch.bfloat16)
        v = torch.as_tensor(_Array(dec, s.v, (pages, heads, hd, PAGE), "<i2"), device="cuda").view(torch.bfloat16)
        return dict(k=k, v=v)
    # INT8 pages: the rows' scales.  Their codes are left out: one that moves to
    # its neighbour with a last bit of the row counts as a wrong whole number.
    # Cleared, as K and V are when the pool is made: unwritten slots are compared too.
    return {n: torch.as_tensor(_Array(dec, getattr(s, n), (pages, heads, PAGE), "<f4"), device="cuda").zero_()
            for n in ("k_scale", "v_scale")}


def _decoder(lib, case, weights, max_seq, batch):
    a = ARCH[case["arch"]]
    cfg = dict(a, max_seq=max_seq, max_batch=batch, wkind=0 if case["kind"] == "int8" else 1,
               kv_kind=_kv_kind(case["kv"]), sparse_k=K_SEL, cand_cap=CAP, rope_len=0, rope_theta=THETA, norm_eps=EPS)
    return be42.Decoder(lib, cfg, weights, _projection(a["head_dim"]))


def prepare(case, seed):
    lib, op = be42.load(), case["op"]
    lib.init()
    s = dict(op=op, lib=lib)
    if op in ("gemv", "gemm", "proj"):
        g, kind, n, k = _gen(seed), case["kind"], case["n"], case["k"]
        s.update(kind=kind, w=_weight(g, n, k, kind))
        if op == "gemv":
            s.update(x=_randn(g, case["batch"], k), y=torch.empty(case["batch"], n, device="cuda"))
        elif op == "gemm":
            s.update(x=_activations(g, case["m"], k), y=torch.empty(case["m"], n, device="cuda"))
        else:
            s.update(w2=_weight(g, n, k, kind), x=_randn(g, case["m"], k))
    elif op == "attn":
        heads, kvh, hd, ctx, batch = (case[n] for n in ("heads", "kv_heads", "head_dim", "ctx", "batch"))
        q = _randn(_gen(seed), batch, heads, hd)
        pool = lib.kv_pool(_kv_kind(case["kv"]), batch, kvh, hd, ctx // PAGE + 1, _projection(hd))
        for b in range(batch):
            pool.append(b, *_history(seed, b, ctx, kvh, hd, q[b]), 0)
        s.update(pool=pool, q=q, scale=1.0 / math.sqrt(hd), out=torch.empty_like(q))
    elif op == "sample":
        g = _gen(seed)
        logits = 2.5 * _randn(g, case["batch"], case["vocab"])
        s.update(logits=logits.to(torch.bfloat16) if case["bf16"] else logits, method=case["method"],
                 u=torch.rand(case["batch"], generator=g, device="cuda"))
    elif op == "step":
        a, batch, ctx = ARCH[case["arch"]], case["batch"], case["ctx"]
        weights, tokens = _model(case, seed), _tokens(case, seed, batch)
        dec = _decoder(lib, case, weights, ctx + 64, batch)
        views = _pool_views(dec)
        # the keys of the prefix follow from the queries of this step, so the
        # step is computed here once, in plain torch, to place them
        _forward(case, seed, weights, tokens, lambda slot, k, v: dec.pool.append(slot, k, v, 0))
        slots, per = a["n_layers"] * batch, -(-ctx // PAGE)
        first, last = dec.pool.s.capacity - slots * per, dec.pool.s.capacity
        # pages are handed out from the highest number down, a slot's prefix at a time
        at = slice(first - slots, first) if ctx % PAGE == 0 else slice(first, last, per)
        s.update(dec=dec, tokens=tokens, pos=ctx, logits=torch.empty(batch, a["vocab"], device="cuda"),
                 cache={n: v[at] for n, v in views.items()})
    else:
        a, n = ARCH[case["arch"]], case["n"]
        dec = _decoder(lib, case, _model(case, seed), -(-n // PAGE) * PAGE, 1)
        s.update(dec=dec, tokens=_tokens(case, seed, n), logits=torch.empty(a["vocab"], device="cuda"),
                 cache=_pool_views(dec), slots=a["n_layers"])
    return s


def run(s):
    lib, op = s["lib"], s["op"]
    if op == "gemv":
        return lib.gemv(*s["w"], s["x"], s["kind"], out=s["y"])
    if op == "gemm":
        xq, sx = (lib.quant_rows_int8 if s["kind"] == "int8" else lib.quant_rows_fp8)(s["x"])
        return dict(xq=xq, sx=sx, y=lib.gemm(xq, sx, *s["w"], s["kind"], out=s["y"]))
    if op == "proj":
        return lib.gemm_f32_multi(s["x"], [s["w"], s["w2"]], s["kind"])
    if op == "attn":
        return lib.lsh_attention(s["pool"], s["q"], K_SEL, CAP, s["scale"], out=s["out"], want_sel=False)[0]
    if op == "sample":
        if s["method"] == "top_p":
            return lib.sample_top_p(s["logits"], 0.8, 0.9, s["u"])
        return lib.sample_temperature(s["logits"], 0.8, s["u"])
    if op == "step":
        s["dec"].step(s["tokens"], s["pos"], logits=s["logits"], sync=False)
        return dict(logits=s["logits"], cache=s["cache"])
    for slot in range(s["slots"]):
        s["dec"].pool.reset(slot)
    s["dec"].prefill(s["tokens"], logits=s["logits"])
    return dict(logits=s["logits"], cache=s["cache"])


# ---- what a pass cannot do without ---------------------------------------------


def _kv_bytes(kv, rows, hd):
    """K and V of `rows` (token, head) rows."""
    return rows * 2 * (hd * 2 if kv == "bf16" else hd + 4)


def _attended(ctx, length):
    """Tokens one query at a `length`-token cache attends to, of a `ctx`-token prefix."""
    pages = -(-length // PAGE)
    return length if pages <= K_SEL else PAGE * min(K_SEL, 2 + int(round(PLANTED * (ctx // PAGE))))


def work(case):
    op = case["op"]
    if op in ("gemv", "gemm", "proj"):
        n, k, m = case["n"], case["k"], case.get("batch", case.get("m"))
        both = 2 if op == "proj" else 1
        codes = (m * k + 4 * m) if op == "gemm" else 0     # the quantized activations are an output too
        return dict(bytes=both * (n * k + 4 * n + 4 * m * n) + 4 * m * k + codes, flops=2.0 * both * m * n * k)
    if op == "attn":
        heads, kvh, hd, ctx, batch = (case[n] for n in ("heads", "kv_heads", "head_dim", "ctx", "batch"))
        rows, pages = _attended(ctx, ctx), -(-ctx // PAGE)
        cand = min(CAP, int(round(PLANTED * (ctx // PAGE)))) if pages > K_SEL else 0
        return dict(bytes=batch * (_kv_bytes(case["kv"], rows * kvh, hd) + cand * 4 * (hd + 1) + 2 * pages + 8 * heads * hd)
                    + 64 * hd, flops=4.0 * batch * heads * rows * hd)
    if op == "sample":
        return dict(bytes=case["batch"] * case["vocab"] * (2 if case["bf16"] else 4), flops=0.0)
    a = ARCH[case["arch"]]
    d, h, kvh, hd, f, vocab, layers = (a[n] for n in ("dim", "n_heads", "n_kv_heads", "head_dim", "hidden_dim", "vocab", "n_layers"))
    shapes = [(h * hd, d), (kvh * hd, d), (kvh * hd, d), (d, h * hd), (f, d), (f, d), (d, f)]
    weights = layers * sum(n * k + 4 * n for n, k in shapes) + vocab * (d + 4)
    macs = layers * sum(n * k for n, k in shapes)
    if op == "step":
        batch, rows = case["batch"], _attended(case["ctx"], case["ctx"] + 1)
        return dict(bytes=weights + batch * (layers * _kv_bytes(case["kv"], (rows + 1) * kvh, hd) + 4 * vocab + d),
                    flops=2.0 * batch * (macs + vocab * d + 2 * layers * h * hd * rows))
    n = case["n"]
    near = min(n, K_SEL * PAGE)      # beyond that, a prompt's tokens attend to few pages
    return dict(bytes=weights + layers * _kv_bytes(case["kv"], n * kvh, hd) + n * d + 4 * vocab,
                flops=2.0 * n * macs + 2.0 * vocab * d + 2.0 * layers * h * hd * near * near)


def tolerance(case):
    """About four times what the path differs by from `exact`, or between two
    evaluations that sum in another order."""
    op = case["op"]
    if op == "sample":
        return "exact"
    if op in ("gemv", "proj"):
        # fp32 activations as fixed-point digits: 2^-24 (INT8) or 1e-6 (FP8) of the largest
        # (measured 1.4e-7, and 5e-6 to 1.2e-5)
        return {"rel": 1e-6 if case["kind"] == "int8" else 5e-5}
    if op == "gemm":
        # measured 4e-8 (whole-number sums) and 2.2e-5 (fp32 sums in the matrix cores)
        return {"rel": 2e-7 if case["kind"] == "int8" else 1e-4, "differ": 0.0}
    if op == "attn":
        return {"rel": 8e-6}     # measured 1.6e-6
    # whole models: a last bit moves a K or V element across a code boundary,
    # and so all that follows (measured 1e-4 to 4e-3)
    return {"rel": 1.5e-2}


# ---- the same in 64 bits -------------------------------------------------------


def _fast_exp(x, nearest=False):
    """Schraudolph's exponential; toward zero, 0 below -87 (attention), or to
    nearest and clamped (SiLU)."""
    bits = 12102203.0 * x.clamp(-87.0, 87.0) + 1065353216.0
    y = (torch.round(bits) if nearest else torch.trunc(bits)).to(torch.int32).view(torch.float32).to(F64)
    return y if nearest else torch.where(x < -87.0, 0.0, y)


def _half_away(x):
    return torch.sign(x) * torch.floor(x.abs() + 0.5)


def _int8_rows(x):
    """Symmetric INT8 codes and scale of the last dimension (fp32 arithmetic)."""
    x = x.to(torch.float32)
    amax = x.abs().amax(-1, keepdim=True)
    some = amax > 0
    code = _half_away(x * torch.where(some, 127.0 / amax, 1.0)).clamp(-127, 127)
    return code, torch.where(some, amax / 127.0, 1.0)


def _fp8_rows(x):
    """E4M3 values (mantissa rounded half up, no carry) and scale of each row."""
    amax = x.abs().amax(-1, keepdim=True)
    s = torch.where(amax > 0, amax / 224.0, 1.0)
    v = (x * (1.0 / s)).to(F64)
    a = v.abs().clamp(max=448.0)
    e = torch.floor(torch.log2(a.clamp(min=1e-30))).clamp(min=-7.0)
    low = e < -6
    unit = torch.exp2(torch.where(low, -6.0, e))
    m = torch.floor(torch.where(low, a / unit, a / unit - 1.0) * 8.0 + 0.5).clamp(max=7.0)
    return torch.sign(v) * unit * torch.where(low, m / 8.0, 1.0 + m / 8.0), s


def _stored(x, kv):
    """K or V rows as the cache holds them: (values, the array that is compared)."""
    if kv == "bf16":
        b = x.to(torch.float32).to(torch.bfloat16)
        return b.to(F64), b
    code, s = _int8_rows(x)
    return code.to(F64) * s.to(F64), s[..., 0]


def _index(k, hp):
    """Head-0 centroid and hash of every full page; k [tokens][kv][hd]."""
    pages = k.shape[0] // PAGE
    c = k[:pages * PAGE, 0].view(pages, PAGE, -1).mean(1)
    return c, ((c @ hp > 0) * (1 << torch.arange(16, device="cuda"))).sum(1).cpu().numpy()


def _push(heap, cap, score, page):
    """A binary min-heap of the best `cap` scores (its array order is the order pages are visited in)."""
    if len(heap) < cap:
        heap.append((score, page))
        i = len(heap) - 1
        while i and heap[(i - 1) // 2][0] > heap[i][0]:
            heap[i], heap[(i - 1) // 2] = heap[(i - 1) // 2], heap[i]
            i = (i - 1) // 2
    elif score > heap[0][0]:
        heap[0], i = (score, page), 0
        while True:
            least = i
            for c in (2 * i + 1, 2 * i + 2):
                if c < len(heap) and heap[c][0] < heap[least][0]:
                    least = c
            if least == i:
                return
            heap[i], heap[least] = heap[least], heap[i]
            i = least


def _route(q, cent, hashes, hp, length):
    """Pages a query visits, in order; q [heads][hd], `length` tokens cached."""
    n = -(-length // PAGE)
    if n <= K_SEL:
        return list(range(n))
    h = int(((q.mean(0) @ hp > 0) * (1 << torch.arange(16, device="cuda"))).sum())
    seen = hashes[:length // PAGE]
    near, found = np.nonzero(np.isin(seen, [h] + [h ^ (1 << b) for b in range(16)]))[0], []
    for probe in [h] + [h ^ (1 << b) for b in range(16)]:
        found += [int(p) for p in near[seen[near] == probe][::-1]]
    middle = [p for p in found[:CAP] if 0 < p < n - 1]
    heap, cap = [], min(K_SEL - 2, len(middle))
    if middle:
        for page, score in zip(middle, (cent[middle] @ q[0]).tolist()):
            _push(heap, cap, score, page)
    return [0, n - 1] + [p for _, p in heap]


def _attend(q, k, v, pages, length):
    """Online softmax of q [T][heads][hd] over k, v [tokens][kv][hd]: query t
    visits pages[t] in order and sees the first length[t] tokens."""
    T, heads, hd = q.shape
    kvh = k.shape[1]
    wide = max(len(p) for p in pages)
    at = torch.tensor([p + [-1] * (wide - len(p)) for p in pages], device="cuda")
    length = torch.tensor(length, device="cuda")
    out = torch.empty(T, heads, hd, dtype=F64, device="cuda")
    for t0 in range(0, T, 64):
        p, ql = at[t0:t0 + 64], q[t0:t0 + 64]
        n = p.shape[0]
        tok = (p[:, :, None] * PAGE + torch.arange(PAGE, device="cuda")).view(n, -1)
        live = ((p >= 0)[:, :, None].expand(-1, -1, PAGE).reshape(n, -1)) & (tok < length[t0:t0 + 64, None])
        tok = tok.clamp(0, k.shape[0] - 1)
        kk, vv = (x[tok].transpose(1, 2).contiguous() for x in (k, v))
        s = torch.matmul(ql.view(n, kvh, -1, hd), kk.transpose(2, 3).contiguous()) / math.sqrt(hd)
        s = torch.where(live[:, None, None], s, -math.inf)
        m = torch.cummax(s, 3).values
        a = _fast_exp(torch.cat([torch.full_like(m[..., :1], -math.inf), m[..., :-1]], 3) - m)
        after = torch.cat([a[..., 1:], torch.ones_like(a[..., :1])], 3).flip(3).cumprod(3).flip(3)
        w = torch.where(live[:, None, None], _fast_exp(s - m) * after, 0.0)
        out[t0:t0 + 64] = (torch.matmul(w, vv) / w.sum(3, keepdim=True)).view(n, heads, hd)
    return out


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w.to(F64)


def _rope(x, pos):
    """x [T][heads][hd] rotated to positions pos (fp32 angles)."""
    half = x.shape[2] // 2
    inv = (1.0 / np.power(np.float32(THETA), np.arange(half, dtype=np.float32) * 2 / np.float32(2 * half))).astype(np.float32)
    ang = torch.from_numpy(np.asarray(pos, np.float32)[:, None] * inv).to("cuda").to(F64)[:, None]
    c, s, x0, x1 = torch.cos(ang), torch.sin(ang), x[..., :half], x[..., half:]
    return torch.cat([x0 * c - x1 * s, x0 * s + x1 * c], 2)


def _forward(case, seed, W, tokens, take=None):
    """The decoder in 64 bits: one token of each of the step's sequences after
    their prefixes, or a prompt's tokens from an empty cache.  Returns the
    logits and each layer's cache rows (step: the page that holds the new
    token); `take` receives every prefix as it is made."""
    a, kind, kv, step = ARCH[case["arch"]], case["kind"], case["kv"], case["op"] == "step"
    heads, kvh, hd = a["n_heads"], a["n_kv_heads"], a["head_dim"]
    hp = torch.from_numpy(_projection(hd)).to("cuda").to(F64)
    T = len(tokens)
    pos = [case["ctx"]] * T if step else list(range(T))
    ids = torch.from_numpy(np.asarray(tokens, np.int64)).to("cuda")
    x = _dense(W["emb"][ids], W["emb_s"][ids], kind)
    cache = []

    def lin(v, one, name):
        return v @ _dense(one["w" + name], one["s" + name], kind).t()

    for l, one in enumerate(W["layers"]):
        h = _rms(x, one["attn_norm"])
        q = _rope(lin(h, one, "q").view(T, heads, hd), pos)
        k = _rope(lin(h, one, "k").view(T, kvh, hd), pos)
        v = lin(h, one, "v").view(T, kvh, hd)
        att = []
        for b in range(T if step else 1):
            rows = slice(b, b + 1) if step else slice(0, T)
            kk, vv = k[rows], v[rows]
            if step:
                slot, ctx = l * T + b, case["ctx"]
                old_k, old_v = _history(seed, slot, ctx, kvh, hd, q[b] if -(-(ctx + 1) // PAGE) > K_SEL else None)
                if take is not None:
                    take(slot, old_k, old_v)
                kk = torch.cat([old_k.view(ctx, kvh, hd).to(F64), kk])
                vv = torch.cat([old_v.view(ctx, kvh, hd).to(F64), vv])
            (kk, kept_k), (vv, kept_v) = _stored(kk, kv), _stored(vv, kv)
            page = case["ctx"] // PAGE * PAGE if step else 0
            cache.append([t[page:].clone() for t in (kept_k, kept_v)])
            cent, hashes = _index(kk, hp)
            where = [_route(q[t], cent, hashes, hp, pos[t] + 1) for t in range(rows.start, rows.stop)]
            att.append(_attend(q[rows], kk, vv, where, [pos[t] + 1 for t in range(rows.start, rows.stop)]))
        x = x + lin(torch.cat(att).view(T, -1), one, "o")
        h = _rms(x, one["ffn_norm"])
        g = lin(h, one, "1")
        x = x + lin(g / (1.0 + _fast_exp(-g, True)) * lin(h, one, "3"), one, "2")
    h = _rms(x if step else x[-1:], W["final_norm"])
    logits = torch.cat([h @ _dense(W["out"][i:i + 16384], W["out_s"][i:i + 16384], kind).t()
                        for i in range(0, a["vocab"], 16384)], 1)
    return logits if step else logits[0], cache


def _paged(rows, pages, turned):
    """Cache rows [slot] of [tokens][kv](...) as `pages` pages a slot in memory
    order (the first page taken has the highest number); turned: the head
    dimension before the tokens."""
    full = []
    for r in rows:
        p = torch.zeros(pages * PAGE, *r.shape[1:], dtype=r.dtype, device="cuda")
        p[:r.shape[0]] = r
        full.append(p.view(pages, PAGE, *r.shape[1:]).transpose(1, 2))
    t = torch.cat(full).flip(0)
    return t.transpose(2, 3) if turned else t


def exact(case, seed):
    op = case["op"]
    if op == "sample":
        return None          # whole numbers
    s = None
    if op in ("gemv", "gemm", "proj"):
        g, kind, n, k = _gen(seed), case["kind"], case["n"], case["k"]
        w, ws = _weight(g, n, k, kind)
        if op == "gemm":
            x = _activations(g, case["m"], k)
            code, sx = _int8_rows(x) if kind == "int8" else _fp8_rows(x)
            x = code.to(F64) * sx.to(F64)
            s = sx[:, 0].to(F64)
        else:
            second = _weight(g, n, k, kind) if op == "proj" else None
            x = _randn(g, case.get("batch", case.get("m")), k).to(F64)
        y = torch.cat([x @ _dense(w[i:i + 16384], ws[i:i + 16384], kind).t() for i in range(0, n, 16384)], 1)
        if op == "gemv":
            return y
        return dict(xq=None, sx=s, y=y) if op == "gemm" else [y, x @ _dense(*second, kind).t()]
    if op == "attn":
        heads, kvh, hd, ctx, batch = (case[n] for n in ("heads", "kv_heads", "head_dim", "ctx", "batch"))
        hp = torch.from_numpy(_projection(hd)).to("cuda").to(F64)
        q = _randn(_gen(seed), batch, heads, hd)
        out = []
        for b in range(batch):
            k, v = (_stored(t.view(ctx, kvh, hd), case["kv"])[0] for t in _history(seed, b, ctx, kvh, hd, q[b]))
            qb = q[b].to(F64)
            out.append(_attend(qb[None], k, v, [_route(qb, *_index(k, hp), hp, ctx)], [ctx]))
        return torch.cat(out)
    step = op == "step"
    n = case["batch"] if step else case["n"]
    logits, cache = _forward(case, seed, _model(case, seed), _tokens(case, seed, n))
    names = ("k", "v") if case["kv"] == "bf16" else ("k_scale", "v_scale")
    pages = 1 if step else -(-n // PAGE)
    if not step and n > 1024:   # such a prompt takes its pages pass by pass
        return dict(logits=logits, cache={m: None for m in names})
    kept = {m: _paged([c[i] for c in cache], pages, m == "v" and case["kv"] == "bf16") for i, m in enumerate(names)}
    return dict(logits=logits, cache=kept)
