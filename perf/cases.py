"""The work whose speed is tracked: the calls that a chunked MTP training run
makes per layer and chunk, through the package's public entry points, over the
sizes such a run meets.

A case is a dict of plain values. ``prepare`` makes what the program has in
hand before the call (inputs, weights, the cached prefix, the chunk's block
mask), ``run`` is one pass, ``exact`` the same outputs in 64 bits by plain
torch. Kinds:

* ``attention`` - one layer's attention of a chunk against the cached prefix:
  the chunk's K/V staged into the cache, the masked attention forward, its
  backward to the chunk's q, k and v.
* ``layer`` - one whole attention block in training: the gated LoRA qkv
  projection, q/k norm + RoPE staged into the cache, attention, the gated LoRA
  output projection; backward to the hidden states and every LoRA matrix.
* ``gated_lora`` - one gated LoRA projection with dropout, forward + backward.
* ``norm_rope`` - q/k norm + RoPE of a chunk with K and V written into the
  cache rows, forward + backward.
* ``soft_ce`` - the sampler's soft cross-entropy, forward + backward, the
  teacher rows a strided view.
* ``bookkeeping`` - everything of a chunk that is not arithmetic: block mask,
  regular-token index and position check, the cache update of each layer, the
  carry-over of the regular rows.
"""
import importlib
import math

import torch

mga = importlib.import_module("mtp-glora_amd")
synthetic = importlib.import_module("mtp-glora_amd.synthetic")

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
QWEN3_VOCAB = 151936
SCALING = 2.0          # alpha / rank
EPS = 1e-6


def _attention(name, n_reg, anchors, draft, pad, prefix, hq=32, hkv=8, d=128, dtype="bf16"):
    c = dict(kind="attention", n_reg=n_reg, anchors=anchors, draft=draft, pad=pad, prefix=prefix, hq=hq, hkv=hkv,
             d=d, dtype=dtype)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the small fp32 decoder of the end-to-end tests (4 query / 2 KV heads
        # of 64): a chunk late in its stream, where launches and latency count
        _attention("attention_small_fp32", 256, 16, 4, 3, 768, hq=4, hkv=2, d=64, dtype="fp32"),
        # the short last chunk that ends a long sequence: few query rows
        # against a long, ragged prefix
        _attention("attention_remainder", 371, 33, 4, 5, 20491),
        # an fp16 run's chunk of odd size in the first part of a sequence
        _attention("attention_fp16_ragged", 1999, 131, 4, 6, 4093, dtype="fp16"),
        # an ordinary chunk of an 8B model: 4096 regular + 256 x 4 mask rows
        _attention("attention_ordinary", 4096, 256, 4, 0, 8192),
        # the last of eight chunks at the same geometry: the long prefix
        _attention("attention_long_prefix", 4096, 512, 4, 0, 28672),
        # one attention block of the 8B model in training, a chunk of a
        # shorter sequence with padding
        dict(name="layer_8b", kind="layer", n_reg=1201, anchors=75, draft=4, pad=35, prefix=4099, hq=32, hkv=8,
             d=128, hidden=4096, rank=32, p=0.05, dtype="bf16"),
        # the fused qkv projection of the ordinary chunk with its dropout
        dict(name="lora_qkv", kind="gated_lora", rows=5120, k=4096, n=6144, rank=96, p=0.05, dtype="bf16"),
        # an output projection over a short odd chunk
        dict(name="lora_o_ragged", kind="gated_lora", rows=1387, k=4096, n=4096, rank=32, p=0.05, dtype="bf16"),
        # q/k norm + RoPE of the ordinary chunk
        dict(name="norm_rope", kind="norm_rope", rows=5120, prefix=8192, hq=32, hkv=8, d=128, dtype="bf16"),
        # the loss over the ordinary chunk's 256 x 4 drafted positions, and
        # over the few of a short chunk
        dict(name="soft_ce_ordinary", kind="soft_ce", rows=1024, vocab=QWEN3_VOCAB, dtype="bf16"),
        dict(name="soft_ce_few_rows", kind="soft_ce", rows=52, vocab=QWEN3_VOCAB, dtype="bf16"),
        # mask, cache updates and carry-over of the ordinary chunk
        dict(name="bookkeeping", kind="bookkeeping", n_reg=4096, anchors=256, draft=4, pad=0, prefix=8192, hkv=8,
             d=128, layers=4, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_chunk(rng, lo, hi):
    """(n_reg, anchors, draft, pad) of a chunk of lo .. hi rows or a few more."""
    n_reg = _log_int(rng, lo, hi)
    draft = rng.choice([2, 4, 4, 4, 8])
    anchors = max(1, int(n_reg * rng.uniform(0.03, 0.13) * 4 / draft))
    return n_reg, anchors, draft, rng.choice([0, 0, rng.randrange(1, 64)])


def draw(rng):
    kind = rng.choice(["attention"] * 5 + ["layer", "gated_lora", "gated_lora", "norm_rope", "soft_ce", "bookkeeping"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    prefix = rng.choice([0, _log_int(rng, 64, 26000), _log_int(rng, 64, 26000), _log_int(rng, 64, 26000)])
    if kind == "attention":
        if rng.random() < 0.15:
            n_reg, anchors, draft, pad = _draw_chunk(rng, 48, 512)
            return _attention(None, n_reg, anchors, draft, pad, min(prefix, _log_int(rng, 64, 2048)), hq=4, hkv=2,
                              d=64, dtype="fp32")
        hq, hkv, d = rng.choice([(32, 8, 128)] * 4 + [(16, 8, 128), (28, 4, 128), (32, 8, 64)])
        n_reg, anchors, draft, pad = _draw_chunk(rng, 96, 4000)
        return _attention(None, n_reg, anchors, draft, pad, prefix, hq=hq, hkv=hkv, d=d, dtype=dtype)
    if kind == "layer":
        n_reg, anchors, draft, pad = _draw_chunk(rng, 128, 3000)
        return dict(kind="layer", n_reg=n_reg, anchors=anchors, draft=draft, pad=pad, prefix=min(prefix, 9000),
                    hq=32, hkv=8, d=128, hidden=4096, rank=rng.choice([16, 32]), p=rng.choice([0.05, 0.1]),
                    dtype="bf16")
    if kind == "gated_lora":
        k, n, mult = rng.choice([(4096, 6144, 3), (4096, 4096, 1), (2560, 6144, 3), (4096, 24576, 2),
                                 (12288, 4096, 1)])
        return dict(kind="gated_lora", rows=_log_int(rng, 96, 6144), k=k, n=n,
                    rank=mult * rng.choice([8, 16, 32]), p=rng.choice([0.0, 0.05, 0.05, 0.1]), dtype="bf16")
    if kind == "norm_rope":
        hq, hkv, d = rng.choice([(32, 8, 128), (32, 8, 128), (16, 8, 128), (4, 2, 64)])
        return dict(kind="norm_rope", rows=_log_int(rng, 64, 6144), prefix=prefix, hq=hq, hkv=hkv, d=d, dtype=dtype)
    if kind == "soft_ce":
        return dict(kind="soft_ce", rows=_log_int(rng, 8, 2048), vocab=rng.choice([QWEN3_VOCAB, QWEN3_VOCAB, 32003]),
                    dtype=rng.choice(["bf16", "bf16", "fp32"]))
    n_reg, anchors, draft, pad = _draw_chunk(rng, 96, 4500)
    return dict(kind="bookkeeping", n_reg=n_reg, anchors=anchors, draft=draft, pad=pad, prefix=prefix, hkv=8, d=128,
                layers=rng.choice([2, 4, 8]), dtype=dtype)


# ---- inputs ---------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, dtype, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda").mul_(scale).to(dtype)


def _chunk(case, seed):
    return synthetic.mtp_chunk(case["n_reg"], synthetic.sample_anchors(case["n_reg"], case["anchors"], seed),
                               case["draft"], pos0=case["prefix"], pad=case["pad"], seed=seed)


def _rows_of(case):
    return case["n_reg"] + case["anchors"] * case["draft"] + case["pad"]


def _attention_inputs(case, seed):
    """Post-norm queries and keys have unit variance per element; q, k, v come
    as transposed views of the projections' [1, S, H, D]."""
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    S, P, hq, hkv, d = _rows_of(case), case["prefix"], case["hq"], case["hkv"], case["d"]
    t = {n: _randn(g, 1, S, h, d, dtype=dt).transpose(1, 2) for n, h in (("q", hq), ("k", hkv), ("v", hkv))}
    t["do"] = _randn(g, 1, S, hq, d, dtype=dt)
    t["kp"], t["vp"] = (_randn(g, 1, hkv, P, d, dtype=dt) for _ in range(2))
    return t


def _lora_inputs(g, k, n, rank, dt):
    return dict(w=_randn(g, n, k, dtype=dt, scale=k ** -0.5), a=_randn(g, rank, k, dtype=dt, scale=k ** -0.5),
                b=_randn(g, n, rank, dtype=dt, scale=0.05))


def _rope_table(pos, d, dt):
    inv = 1e6 ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float32) / d)
    ang = pos.float()[:, None] * inv
    ang = torch.cat([ang, ang], dim=-1)
    return ang.cos().to(dt)[None], ang.sin().to(dt)[None]


def _norm_rope_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    S, hq, hkv, d = case["rows"], case["hq"], case["hkv"], case["d"]
    qkv = _randn(g, 1, S, (hq + 2 * hkv) * d, dtype=dt)      # the fused projection's output
    q, k, v = (x.view(1, S, -1, d) for x in qkv.split([hq * d, hkv * d, hkv * d], dim=-1))
    cos, sin = _rope_table(case["prefix"] + torch.arange(S, device="cuda"), d, dt)
    return dict(q=q, k=k, v=v, qw=(1 + 0.1 * _randn(g, d, dtype=torch.float32)).to(dt),
                kw=(1 + 0.1 * _randn(g, d, dtype=torch.float32)).to(dt), cos=cos, sin=sin,
                gq=_randn(g, 1, hq, S, d, dtype=dt), gk=_randn(g, 1, hkv, S, d, dtype=dt),
                gv=_randn(g, 1, hkv, S, d, dtype=dt))


def _gated_lora_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    t = _lora_inputs(g, case["k"], case["n"], case["rank"], dt)
    t["x"] = _randn(g, 1, case["rows"], case["k"], dtype=dt)
    t["dy"] = _randn(g, 1, case["rows"], case["n"], dtype=dt)
    t["gate"] = (torch.rand(1, case["rows"], 1, generator=g, device="cuda") < 0.2).long()
    t["seed"] = 1000003 * (seed + 1)
    return t


def _layer_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    S, P, hq, hkv, d, hid = _rows_of(case), case["prefix"], case["hq"], case["hkv"], case["d"], case["hidden"]
    chunk = _chunk(case, seed)
    t = dict(chunk=chunk, x=_randn(g, 1, S, hid, dtype=dt), dy=_randn(g, 1, S, hid, dtype=dt),
             qkv=_lora_inputs(g, hid, (hq + 2 * hkv) * d, 3 * case["rank"], dt),
             o=_lora_inputs(g, hq * d, hid, case["rank"], dt),
             qw=(1 + 0.1 * _randn(g, d, dtype=torch.float32)).to(dt),
             kw=(1 + 0.1 * _randn(g, d, dtype=torch.float32)).to(dt),
             kp=_randn(g, 1, hkv, P, d, dtype=dt), vp=_randn(g, 1, hkv, P, d, dtype=dt),
             gate=chunk["gate_mask"].clamp(min=0)[:, :, None], seed=1000003 * (seed + 1))
    t["cos"], t["sin"] = _rope_table(chunk["position_ids"][0], d, dt)
    return t


def _soft_ce_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    n, v = case["rows"], case["vocab"]
    x = _randn(g, 1, n, v, dtype=dt, scale=2.0)
    full = torch.empty(1, 2 * n, v, device="cuda", dtype=dt)   # the teacher's rows lie among others
    full[:, 1::2] = 0
    full[:, ::2] = x + _randn(g, 1, n, v, dtype=dt)
    return dict(x=x, full=full)


def _cache(kp, vp, rows, layers=1):
    hkv, P, d = kp.shape[1:]
    cache = mga.StreamingKVCache(capacity=P + rows, num_layers=layers, num_kv_heads=hkv, head_dim=d, dtype=kp.dtype,
                                 device=kp.device)
    if P:
        cache.append_prefix([kp] * layers, [vp] * layers)
    return cache


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, case=case)
    if kind == "attention":
        t = _attention_inputs(case, seed)
        chunk = _chunk(case, seed)
        s.update(q=t["q"].requires_grad_(), k=t["k"].requires_grad_(), v=t["v"].requires_grad_(), do=t["do"],
                 cache=_cache(t["kp"], t["vp"], _rows_of(case)),
                 mask=mga.build_mtp_block_mask(chunk["gate_mask"], case["prefix"]), module=torch.nn.Module())
    elif kind == "layer":
        t = _layer_inputs(case, seed)
        for p in (t["x"], t["qkv"]["a"], t["qkv"]["b"], t["o"]["a"], t["o"]["b"]):
            p.requires_grad_()
        s.update(t, cache=_cache(t["kp"], t["vp"], _rows_of(case)),
                 mask=mga.build_mtp_block_mask(t["chunk"]["gate_mask"], case["prefix"]), module=torch.nn.Module())
    elif kind == "gated_lora":
        t = _gated_lora_inputs(case, seed)
        for n in ("x", "a", "b"):
            t[n].requires_grad_()
        s.update(t)
    elif kind == "norm_rope":
        t = _norm_rope_inputs(case, seed)
        for n in ("q", "k", "v"):
            t[n] = t[n].detach().requires_grad_()
        cache = mga.StreamingKVCache(capacity=case["prefix"] + case["rows"], num_layers=1, num_kv_heads=case["hkv"],
                                     head_dim=case["d"], dtype=DTYPES[case["dtype"]], device=t["q"].device)
        cache.prefix_len = case["prefix"]
        s.update(t, cache=cache)
    elif kind == "soft_ce":
        t = _soft_ce_inputs(case, seed)
        s.update(x=t["x"].requires_grad_(), teacher=t["full"][:, ::2])
    else:
        g, dt = _gen(seed), DTYPES[case["dtype"]]
        S, P, hkv, d, layers = _rows_of(case), case["prefix"], case["hkv"], case["d"], case["layers"]
        mgr = mga.StreamingKVCacheManager(capacity=P + S)
        mgr.past_seen_tokens = P
        mgr.cache = _cache(_randn(g, 1, hkv, P, d, dtype=dt), _randn(g, 1, hkv, P, d, dtype=dt), S, layers)
        kv = [tuple(_randn(g, 1, S, hkv, d, dtype=dt).transpose(1, 2) for _ in range(2)) for _ in range(layers)]
        s.update(mgr=mgr, kv=kv, chunk=_chunk(case, seed))
    return s


# ---- one pass ---------------------------------------------------------------

def _run_layer(s):
    c = s["case"]
    S, hq, hkv, d = _rows_of(c), c["hq"], c["hkv"], c["d"]
    w, wo = s["qkv"], s["o"]
    qkv = mga.gated_lora_linear(s["x"], w["w"], w["a"], w["b"], s["gate"], SCALING, c["p"], s["seed"])
    q, k, v = (x.view(1, S, -1, d) for x in qkv.split([hq * d, hkv * d, hkv * d], dim=-1))
    q, k, v = importlib.import_module("mtp-glora_amd.rope").qk_norm_rope_stage(
        q, k, v, s["qw"], s["kw"], s["cos"], s["sin"], EPS, s["cache"], 0)
    k, v = s["cache"].update(k, v, 0)
    o, _ = mga.mtp_attention_forward(s["module"], q, k, v, s["mask"], scaling=d ** -0.5)
    y = mga.gated_lora_linear(o.reshape(1, S, hq * d), wo["w"], wo["a"], wo["b"], s["gate"], SCALING, c["p"],
                              s["seed"] + 1)
    return (y, *torch.autograd.grad(y, [s["x"], w["a"], w["b"], wo["a"], wo["b"]], s["dy"]))


def run(s):
    kind, c = s["kind"], s["case"]
    if kind == "attention":
        k, v = s["cache"].update(s["k"], s["v"], 0)
        o, lse = mga.mtp_attention_forward(s["module"], s["q"], k, v, s["mask"], scaling=c["d"] ** -0.5)
        return (o, lse, *torch.autograd.grad(o, [s["q"], s["k"], s["v"]], s["do"]))
    if kind == "layer":
        return _run_layer(s)
    if kind == "gated_lora":
        y = mga.gated_lora_linear(s["x"], s["w"], s["a"], s["b"], s["gate"], SCALING, c["p"], s["seed"])
        return (y, *torch.autograd.grad(y, [s["x"], s["a"], s["b"]], s["dy"]))
    if kind == "norm_rope":
        q, k, v = importlib.import_module("mtp-glora_amd.rope").qk_norm_rope_stage(
            s["q"], s["k"], s["v"], s["qw"], s["kw"], s["cos"], s["sin"], EPS, s["cache"], 0)
        return (q, k, v, *torch.autograd.grad([q, k, v], [s["q"], s["k"], s["v"]], [s["gq"], s["gk"], s["gv"]]))
    if kind == "soft_ce":
        loss = mga.StableSoftCrossEntropy.apply(s["x"], s["teacher"])
        return (loss, *torch.autograd.grad(loss, [s["x"]]))
    mgr, P = s["mgr"], c["prefix"]
    chunk = mgr.prepare_data_with_kv_cache(dict(s["chunk"]))
    cache = mgr.cache
    for i, (k, v) in enumerate(s["kv"]):
        cache.update(k, v, i)
    cache = mgr.extract_regular_kv_cache_for_next_chunk(chunk, cache)
    seen = mgr.past_seen_tokens
    rows = [tuple(t[:, :, P:] for t in kv) for kv in cache]
    cache.crop(P)                       # the next pass streams the same chunk
    mgr.past_seen_tokens = P
    m = chunk["attention_mask"]
    return dict(seen=seen, gate=chunk["gate_mask"], code=m.mtp_code, rows=rows, kv_num=m.kv_num_blocks,
                kv_idx=m.kv_indices, full_kv_num=m.full_kv_num_blocks, full_kv_idx=m.full_kv_indices,
                q_num=m.q_num_blocks, q_idx=m.q_indices, full_q_num=m.full_q_num_blocks,
                full_q_idx=m.full_q_indices)


# ---- what a pass cannot do without --------------------------------------------

def _attention_work(c, eb):
    """Products over the pairs the mask allows: forward 2, backward 3 (5 where
    the key has a gradient), of 2 D flops each; a block's masks see the
    regular tokens up to their anchor and the block itself."""
    S, P, hq, hkv, d = _rows_of(c), c["prefix"], c["hq"], c["hkv"], c["d"]
    n, a, k = c["n_reg"], c["anchors"], c["draft"]
    pre = (n + a * k) * P
    cur = n * (n + 1) / 2 + a * k * n / 2 + a * k * (k + 1) / 2
    flops = hq * d * (10 * pre + 14 * cur)
    by = eb * d * (4 * S * hq + 4 * S * hkv + 2 * P * hkv) + 4 * hq * S
    return by, flops


def work(case):
    kind, eb = case["kind"], 4 if case["dtype"] == "fp32" else 2
    if kind == "attention":
        by, fl = _attention_work(case, eb)
        return dict(bytes=by, flops=fl)
    if kind == "layer":
        S, hid, nq, r = _rows_of(case), case["hidden"], (case["hq"] + 2 * case["hkv"]) * case["d"], case["rank"]
        no = case["hq"] * case["d"]
        by = eb * (4 * S * hid + nq * hid + no * hid + 2 * 3 * r * (hid + nq) + 2 * r * (hid + no)
                   + 2 * case["prefix"] * case["hkv"] * case["d"])
        fl = _attention_work(case, eb)[1] + 4 * S * hid * (nq + no) + 6 * S * (3 * r * (hid + nq) + r * (hid + no))
        return dict(bytes=by, flops=fl)
    if kind == "gated_lora":
        S, k, n, r = case["rows"], case["k"], case["n"], case["rank"]
        return dict(bytes=eb * (2 * S * k + 2 * S * n + k * n + 2 * r * (k + n)), flops=4 * S * k * n + 6 * S * r * (k + n))
    if kind == "norm_rope":
        S, hq, hkv, d = case["rows"], case["hq"], case["hkv"], case["d"]
        return dict(bytes=eb * S * d * (4 * hq + 4 * hkv + 4 * hkv + 2), flops=40 * S * d * (hq + hkv))
    if kind == "soft_ce":
        return dict(bytes=3 * eb * case["rows"] * case["vocab"], flops=16 * case["rows"] * case["vocab"])
    S, R, P = _rows_of(case), case["n_reg"], case["prefix"]
    nq, nkv = -(-S // 128), -(-(P + S) // 128)
    return dict(bytes=case["layers"] * 4 * eb * (S + R) * case["hkv"] * case["d"] + 32 * S + 16 * nq * nkv,
                flops=S * nkv)


def tolerance(case):
    kind, dt = case["kind"], case["dtype"]
    if kind == "bookkeeping":
        return "exact"
    if kind == "soft_ce":
        return {"rel": 1e-5 if dt == "fp32" else 8e-3}
    if kind == "norm_rope":       # roundings after each step of the 16-bit forward
        return {"rel": 1.2e-2 if dt == "bf16" else 1.5e-3}
    if dt == "fp32":
        return {"rel": 1e-5}
    return {"rel": 1.2e-2 if dt == "bf16" else 2e-3}


# ---- the same outputs in 64 bits ------------------------------------------------

def _allowed(gate, P):
    """[S, P + S] truth values of the MTP mask: a key is seen when it does not
    follow the query and is a regular token or of the query's own block; a
    padding query sees nothing."""
    S = gate.numel()
    code = torch.where(gate == 0, -2, P + torch.cumsum((gate == 0).long(), 0))
    code = torch.where(gate == -1, -1, code)
    keys = torch.cat([torch.full((P,), -2, device=gate.device, dtype=code.dtype), code])
    qi = torch.arange(S, device=gate.device)[:, None] + P
    ki = torch.arange(P + S, device=gate.device)[None]
    return (qi >= ki) & (code != -1)[:, None] & ((keys == -2)[None] | (keys[None] == code[:, None]))


class _Attend(torch.autograd.Function):
    """q [Hq, S, D], k and v [Hkv, L, D], a head at a time; gradients of the keys
    from ``P`` on."""

    @staticmethod
    def forward(ctx, q, k, v, allowed, P, scale):
        g = q.shape[0] // k.shape[0]
        o, lse = torch.empty_like(q), torch.empty(q.shape[:2], device=q.device, dtype=q.dtype)
        for h in range(q.shape[0]):
            s = (q[h] @ k[h // g].t()).mul_(scale).masked_fill_(~allowed, -math.inf)
            lse[h] = torch.logsumexp(s, dim=-1)
            p = s.sub_(lse[h][:, None]).exp_().nan_to_num_(nan=0.0)
            o[h] = p @ v[h // g]
        ctx.save_for_backward(q, k, v, allowed, o, lse)
        ctx.P, ctx.scale = P, scale
        return o, lse

    @staticmethod
    def backward(ctx, do, _):
        q, k, v, allowed, o, lse = ctx.saved_tensors
        P, g = ctx.P, q.shape[0] // k.shape[0]
        dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
        for h in range(q.shape[0]):
            j = h // g
            p = (q[h] @ k[j].t()).mul_(ctx.scale).masked_fill_(~allowed, -math.inf)
            p = p.sub_(lse[h][:, None]).exp_().nan_to_num_(nan=0.0)
            dv[j, P:] += p[:, P:].t() @ do[h]
            ds = (do[h] @ v[j].t()).sub_((do[h] * o[h]).sum(-1, keepdim=True)).mul_(p).mul_(ctx.scale)
            dq[h] = ds @ k[j]
            dk[j, P:] += ds[:, P:].t() @ q[h]
        return dq, dk, dv, None, None, None


def _fmix32(h):
    m = 0xFFFFFFFF
    h = h ^ (h >> 16)
    h = (h * 0x85EBCA6B) & m
    h = h ^ (h >> 13)
    h = (((h & 0xFFFF) * 0xC2B2AE35) + (((h >> 16) * 0xC2B2AE35 & 0xFFFF) << 16)) & m
    return h ^ (h >> 16)


def _keep(S, k, p, seed):
    """The dropout's keep mask of an [S, k] input: a counter hash of the seed and
    the element pair (16 bits an element)."""
    j = torch.arange(S * k // 2, device="cuda", dtype=torch.int64)
    h = _fmix32((j & 0xFFFFFFFF) ^ (seed & 0xFFFFFFFF))
    h = _fmix32(h ^ (j >> 32) ^ (seed >> 32))
    thr = round(p * 65536)
    return torch.stack([(h & 0xFFFF) >= thr, (h >> 16) >= thr], dim=-1).view(S, k)


def _lora_exact(x, w, a, b, gate, p, seed):
    h = x * _keep(*x.shape, p, seed) / (1 - p) if p > 0 else x
    return x @ w.t() + SCALING * ((h @ a.t()) @ b.t()) * gate


def _norm_rope_exact(x, w, cos, sin):
    """x [S, H, D] -> [H, S, D]."""
    n = w * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    half = x.shape[-1] // 2
    rot = torch.cat([-n[..., half:], n[..., :half]], dim=-1)
    return (n * cos[:, None] + rot * sin[:, None]).transpose(0, 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "bookkeeping":
        return None
    if kind == "attention":
        t = {n: x.double()[0] for n, x in _attention_inputs(case, seed).items()}
        allowed = _allowed(_chunk(case, seed)["gate_mask"][0], case["prefix"])
        q, k, v = (t[n].requires_grad_() for n in ("q", "k", "v"))
        o, lse = _Attend.apply(q, torch.cat([t["kp"], k], 1), torch.cat([t["vp"], v], 1), allowed, case["prefix"],
                               case["d"] ** -0.5)
        o = o.transpose(0, 1)
        return (o[None], lse[None], *(g[None] for g in torch.autograd.grad(o, [q, k, v], t["do"])))
    if kind == "gated_lora":
        t = _gated_lora_inputs(case, seed)
        x, w, a, b, dy, gate = (t[n].double() for n in ("x", "w", "a", "b", "dy", "gate"))
        for p in (x, a, b):
            p.requires_grad_()
        y = _lora_exact(x[0], w, a, b, gate[0], case["p"], t["seed"])[None]
        return (y, *torch.autograd.grad(y, [x, a, b], dy))
    if kind == "norm_rope":
        t = {n: x.double() for n, x in _norm_rope_inputs(case, seed).items()}
        q, k, v = (t[n].requires_grad_() for n in ("q", "k", "v"))
        qe = _norm_rope_exact(q[0], t["qw"], t["cos"][0], t["sin"][0])[None]
        ke = _norm_rope_exact(k[0], t["kw"], t["cos"][0], t["sin"][0])[None]
        ve = v.transpose(1, 2)
        return (qe, ke, ve, *torch.autograd.grad([qe, ke, ve], [q, k, v], [t["gq"], t["gk"], t["gv"]]))
    if kind == "soft_ce":
        t = _soft_ce_inputs(case, seed)
        loss, grad = 0.0, torch.empty(t["x"].shape, device="cuda", dtype=torch.float64)
        for i in range(0, case["rows"], 64):
            x, y = t["x"][:, i:i + 64].double(), t["full"][:, ::2][:, i:i + 64].double()
            lx, py = torch.log_softmax(x, -1), torch.softmax(y, -1)
            loss = loss - (py * lx).sum()
            grad[:, i:i + 64] = lx.exp() - py
        return loss, grad
    t = _layer_inputs(case, seed)
    S, P, hq, hkv, d = _rows_of(case), case["prefix"], case["hq"], case["hkv"], case["d"]
    x, dy, kp, vp, qw, kw, cos, sin, gate = (t[n].double() for n in ("x", "dy", "kp", "vp", "qw", "kw", "cos", "sin",
                                                                     "gate"))
    w, wo = ({n: m.double() for n, m in t[i].items()} for i in ("qkv", "o"))
    for p in (x, w["a"], w["b"], wo["a"], wo["b"]):
        p.requires_grad_()
    qkv = _lora_exact(x[0], w["w"], w["a"], w["b"], gate[0], case["p"], t["seed"])
    q, k, v = (m.view(S, -1, d) for m in qkv.split([hq * d, hkv * d, hkv * d], dim=-1))
    q, k = _norm_rope_exact(q, qw, cos[0], sin[0]), _norm_rope_exact(k, kw, cos[0], sin[0])
    o, _ = _Attend.apply(q, torch.cat([kp[0], k], 1), torch.cat([vp[0], v.transpose(0, 1)], 1),
                         _allowed(t["chunk"]["gate_mask"][0], P), P, d ** -0.5)
    o = o.transpose(0, 1).reshape(S, hq * d)
    y = _lora_exact(o, wo["w"], wo["a"], wo["b"], gate[0], case["p"], t["seed"] + 1)[None]
    return (y, *torch.autograd.grad(y, [x, w["a"], w["b"], wo["a"], wo["b"]], dy))
