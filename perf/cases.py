"""The attention work a serving program has this package do, as cases that can be timed
and checked.

Layouts are those of the models the package serves: Qwen3-0.6B (16 query heads over 8 KV
heads), Qwen3-8B (32 over 8), the Qwen2.5-VL decoder (28 over 4) and its vision tower (16
heads of 80).  Lengths come from the case's own ``lens_seed`` (so that the work of a case is
known without its inputs); values, block tables and weights from the seed of ``prepare``.
Keys and queries are N(0, 1), as rows behind a QK norm are.  Paged pools are scattered over
a shuffled block list and filled throughout, so that a wrong table entry shows.

Kinds of cases:
  decode    one new token of every sequence against its paged keys
  prefill   packed causal attention over fresh keys
  chunked   query chunks after cached context, over the paged cache
  vision    non-causal packed attention, one chunk per image or per window
  rope      QK norm, rotary embedding and the cache write of a step's new tokens
  layer     a decoder layer's whole attention module on a step of decodes and chunks
"""
from __future__ import annotations

import math

import torch

from nano_inference_amd import PagedCausalSelfAttention, ops, window_index
from nano_inference_amd.context import PackedAttentionMetadata

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp8": torch.bfloat16, "f32": torch.float32}
LAYOUTS = {"qwen3_0p6b": (16, 8), "qwen3_8b": (32, 8), "qwen25vl": (28, 4)}
HIDDEN = {"qwen3_0p6b": 1024, "qwen3_8b": 4096}
D = 128
EPS = 1e-6
ROPE_BASE = 1e6


def listed():
    return [
        # One user typing: a single sequence decodes; latency and launches are all of it.
        dict(name="decode_one", kind="decode", layout="qwen3_0p6b", store="bf16", batch=1,
             lo=1023, hi=1023, block=16, lens_seed=11),
        # A full server step of the 8B model: the headline decode.
        dict(name="decode_qwen3_8b", kind="decode", layout="qwen3_8b", store="bf16", batch=64,
             lo=512, hi=8192, block=16, lens_seed=2002),
        # The same step over an fp8 cache.
        dict(name="decode_fp8", kind="decode", layout="qwen3_8b", store="fp8", batch=64,
             lo=512, hi=8192, block=16, lens_seed=2002),
        # The engine's default float32 on the small model, a few users.
        dict(name="decode_f32", kind="decode", layout="qwen3_0p6b", store="f32", batch=16,
             lo=256, hi=2304, block=16, lens_seed=1001),
        # A prefill-first step: eight prompts together.
        dict(name="prefill_qwen3_8b", kind="prefill", layout="qwen3_8b", store="bf16", batch=8,
             lo=256, hi=4096, lens_seed=3003),
        # One prompt of odd length alone: the time to a first token.
        dict(name="prefill_one", kind="prefill", layout="qwen3_8b", store="bf16", batch=1,
             lo=1531, hi=1531, lens_seed=12),
        # The engine's default float32: a few short prompts on the small model.
        dict(name="prefill_f32", kind="prefill", layout="qwen3_0p6b", store="f32", batch=4,
             lo=128, hi=1024, lens_seed=13),
        # Chunked prefill of eight long prompts over an fp8 cache.
        dict(name="chunked_fp8", kind="chunked", layout="qwen3_8b", store="fp8", batch=8,
             chunk=512, lo=0, hi=8192, block=16, lens_seed=3103),
        # The vision tower's full-attention blocks on four images of mixed sizes.
        dict(name="vision_full", kind="vision", window=False,
             grids="28x28,36x52,64x48,20x90"),
        # Its windowed blocks (28 of 32) on the same images.
        dict(name="vision_window", kind="vision", window=True,
             grids="28x28,36x52,64x48,20x90"),
        # The step before the attention at the scheduler's full 8192-token step.
        dict(name="rope_8192", kind="rope", layout="qwen3_8b", store="bf16", tokens=8192,
             norm=True, mrope=False, block=16),
        # A mixed step through the drop-in layer: 24 users decode while one long prompt
        # (the scheduler's 1024-token chunk after about 12k cached tokens) streams in.
        dict(name="layer_mixed", kind="layer", layout="qwen3_8b", batch=24, lo=512, hi=6144,
             chunk=1024, prior=12305, block=16, lens_seed=14),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw(rng):
    kind = rng.choice(["decode", "decode", "decode_f32", "prefill", "prefill_f32", "chunked",
                       "chunked", "vision", "rope", "layer"])
    seed = rng.randrange(1 << 20)
    layout = rng.choice(["qwen3_0p6b", "qwen3_8b", "qwen3_8b", "qwen25vl"])
    block = rng.choice([16, 16, 32])
    if kind in ("decode", "decode_f32"):
        f32 = kind == "decode_f32"
        hi = _log_int(rng, 48, 4096 if f32 else 8192)
        return dict(kind="decode", layout="qwen3_0p6b" if f32 else layout,
                    store="f32" if f32 else rng.choice(["bf16", "bf16", "fp8"]),
                    batch=_log_int(rng, 1, 32 if f32 else 64), lo=max(1, hi // 16), hi=hi,
                    block=16 if f32 else block, lens_seed=seed)
    if kind in ("prefill", "prefill_f32"):
        f32 = kind == "prefill_f32"
        hi = _log_int(rng, 24, 1024 if f32 else 4096)
        return dict(kind="prefill", layout="qwen3_0p6b" if f32 else layout,
                    store="f32" if f32 else "bf16", batch=_log_int(rng, 1, 4 if f32 else 8),
                    lo=max(1, hi // 8), hi=hi, lens_seed=seed)
    if kind == "chunked":
        hi = _log_int(rng, 64, 16384)
        return dict(kind="chunked", layout=layout, store=rng.choice(["bf16", "bf16", "fp8"]),
                    batch=_log_int(rng, 1, 8), chunk=_log_int(rng, 24, 1024), lo=hi // 4, hi=hi,
                    block=block, lens_seed=seed)
    if kind == "vision":
        grids = ["%dx%d" % (2 * rng.randint(6, 32), 2 * rng.randint(6, 32))
                 for _ in range(rng.randint(1, 4))]
        return dict(kind="vision", window=rng.random() < 0.6, grids=",".join(grids))
    if kind == "rope":
        mrope = layout == "qwen25vl"
        return dict(kind="rope", layout=layout, store=rng.choice(["bf16", "bf16", "fp8", "f32"]),
                    tokens=_log_int(rng, 1, 8192), norm=not mrope, mrope=mrope, block=block)
    hi = _log_int(rng, 64, 6144)
    return dict(kind="layer", layout=rng.choice(["qwen3_0p6b", "qwen3_8b"]),
                batch=_log_int(rng, 1, 32), lo=max(1, hi // 8), hi=hi,
                chunk=_log_int(rng, 16, 1024), prior=_log_int(rng, 1, 12288), block=block,
                lens_seed=seed)


def _cost(case):
    w = work(case)
    # fp32 scores are summed in 64 bits, at a thirtieth of the 16-bit rate
    return max(w["bytes"], w["flops"] / (8 if case.get("store") == "f32" else 300))


def draw(rng):
    cap = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= cap:
            return case


# ---- lengths ---------------------------------------------------------------------------


def _lens(case):
    g = torch.Generator("cpu")
    g.manual_seed(case["lens_seed"])
    return torch.randint(case["lo"], case["hi"] + 1, (case["batch"],), generator=g).tolist()


def _grids(case):
    return [(1, *map(int, s.split("x"))) for s in case["grids"].split(",")]


def _vision_lens(case):
    if case["window"]:
        cu = window_index(_grids(case))[1].tolist()
        return [b - a for a, b in zip(cu[:-1], cu[1:])]
    return [h * w for _, h, w in _grids(case)]


# ---- inputs ----------------------------------------------------------------------------


class _Values:
    """N(0, 1) tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(DEV)
        self.g.manual_seed(seed)
        self.cpu = torch.Generator("cpu")
        self.cpu.manual_seed(seed + 1)

    def normal(self, *shape, dtype=torch.bfloat16, scale=1.0):
        x = torch.randn(shape, generator=self.g, device=DEV, dtype=dtype)
        return x if scale == 1.0 else x.mul_(scale)

    def tables(self, ctx, block):
        """Shuffled block tables of sequences of ``ctx`` tokens; the pool's block count."""
        n = [-(-c // block) for c in ctx]
        pool = sum(n) + 64
        perm = torch.randperm(pool, generator=self.cpu).to(torch.int32)
        t = torch.zeros((len(ctx), max(n)), dtype=torch.int32)
        at = 0
        for i, k in enumerate(n):
            t[i, :k] = perm[at:at + k]
            at += k
        return t, pool


def _fp8_rows(x):
    """e4m3 codes (as bytes) and row scales max |x| / 448 of the rows of x."""
    s = x.float().abs().amax(dim=-1) / 448.0
    codes = (x.float() / s.unsqueeze(-1)).to(torch.float8_e4m3fn)
    return codes.view(torch.uint8), s


def _pool(v, store, hkv, block, blocks):
    """(k_cache, v_cache, k_scale, v_scale) of one layer, filled."""
    k, w = (v.normal(blocks, hkv, block, D, dtype=DTYPES[store]) for _ in range(2))
    if store != "fp8":
        return k, w, None, None
    (kc, ks), (vc, vs) = _fp8_rows(k), _fp8_rows(w)
    return kc, vc, ks, vs


def prepare(case, seed):
    v = _Values(seed)
    kind = case["kind"]
    if kind == "vision":
        lens = _vision_lens(case)
        q, k, w = (v.normal(sum(lens), 16, 80) for _ in range(3))
        return dict(kind=kind, q=q, k=k, v=w, cu=_cu(lens), longest=max(lens))
    h, hkv = LAYOUTS[case["layout"]]
    if kind == "prefill":
        lens, dt = _lens(case), DTYPES[case["store"]]
        q, k, w = (v.normal(sum(lens), n, D, dtype=dt) for n in (h, hkv, hkv))
        return dict(kind=kind, q=q, k=k, v=w, cu=_cu(lens), longest=max(lens))
    if kind == "rope":
        return _prepare_rope(case, v, h, hkv)
    if kind == "layer":
        return _prepare_layer(case, v, h, hkv)
    lens = _lens(case)
    if kind == "chunked":
        lens = [n + case["chunk"] for n in lens]
    tables, blocks = v.tables(lens, case["block"])
    kc, vc, ks, vs = _pool(v, case["store"], hkv, case["block"], blocks)
    rows = case["batch"] * case.get("chunk", 1)
    s = dict(kind=kind, q=v.normal(rows, h, D, dtype=DTYPES[case["store"]]), k_cache=kc,
             v_cache=vc, k_scale=ks, v_scale=vs, tables=tables.to(DEV),
             ctx=torch.tensor(lens, dtype=torch.int64, device=DEV))
    if kind == "chunked":
        c = case["chunk"]
        s["q_start"] = torch.arange(case["batch"], dtype=torch.int32, device=DEV) * c
        s["q_len"] = torch.full((case["batch"],), c, dtype=torch.int32, device=DEV)
        s["longest"] = c
    return s


def _cu(lens):
    return torch.tensor([0] + lens, dtype=torch.int64).cumsum(0).to(torch.int32).to(DEV)


def _inv_freq():
    return 1.0 / (ROPE_BASE ** (torch.arange(0, D, 2, dtype=torch.float32) / D))


MROPE = (16, 24, 24)


def _prepare_rope(case, v, h, hkv):
    t, dt = case["tokens"], DTYPES[case["store"]]
    blocks = -(-t // case["block"]) + 64
    perm = torch.randperm(blocks * case["block"], generator=v.cpu)[:t]
    # prompts of up to 8k tokens: positions anywhere below, mRoPE axes apart
    shape = (3, t) if case["mrope"] else (t,)
    pos = torch.randint(0, 8192, shape, generator=v.cpu)
    kc, vc, ks, vs = _pool(v, case["store"], hkv, case["block"], blocks)
    weight = lambda: (1 + v.normal(D, dtype=torch.float32, scale=0.1)).to(dt)  # noqa: E731
    return dict(kind="rope", q=v.normal(t, h, D, dtype=dt), k=v.normal(t, hkv, D, dtype=dt),
                v=v.normal(t, hkv, D, dtype=dt),
                qw=weight() if case["norm"] else None, kw=weight() if case["norm"] else None,
                pos=pos.to(DEV), inv=_inv_freq().to(DEV),
                section=MROPE if case["mrope"] else None,
                k_cache=kc, v_cache=vc, k_scale=ks, v_scale=vs, slots=perm.to(DEV))


def _prepare_layer(case, v, h, hkv):
    hidden, chunk, block = HIDDEN[case["layout"]], case["chunk"], case["block"]
    attn = PagedCausalSelfAttention(hidden, h, hkv, D, use_qk_norm=True, rope_base=ROPE_BASE)
    attn = attn.to(device=DEV, dtype=torch.bfloat16).requires_grad_(False)
    attn.layer_idx = 0
    for name, p in attn.named_parameters():
        if p.dim() == 2:  # outputs about as large as inputs
            p.copy_(v.normal(*p.shape, scale=p.shape[1] ** -0.5))
        else:
            p.copy_(1 + v.normal(*p.shape, scale=0.1))
    dec = _lens(case)
    ctx = dec + [case["prior"] + chunk]
    tables, blocks = v.tables(ctx, block)
    kc, vc, _, _ = _pool(v, "bf16", hkv, block, blocks)
    pos = torch.tensor([n - 1 for n in dec] + list(range(case["prior"], case["prior"] + chunk)))
    row = torch.tensor(list(range(len(dec))) + [len(dec)] * chunk)
    slots = tables[row, pos // block].long() * block + pos % block
    n = len(dec)
    md = PackedAttentionMetadata(
        context_lens=torch.tensor(ctx, dtype=torch.int64, device=DEV),
        kv_block_tables=tables.to(DEV), slot_mapping=slots.unsqueeze(0).to(DEV),
        k_cache=kc.unsqueeze(0), v_cache=vc.unsqueeze(0),
        q_start=torch.arange(n + 1, dtype=torch.int32, device=DEV),
        q_len=torch.tensor([1] * n + [chunk], dtype=torch.int32, device=DEV),
        num_decode=n, max_q_len=chunk)
    return dict(kind="layer", attn=attn, x=v.normal(1, n + chunk, hidden),
                pos=pos.unsqueeze(0).to(DEV), md=md)


# ---- one pass --------------------------------------------------------------------------


def run(s):
    kind = s["kind"]
    if kind == "decode":
        return ops.paged_decode(s["q"], s["k_cache"], s["v_cache"], s["tables"], s["ctx"],
                                k_scale=s["k_scale"], v_scale=s["v_scale"])
    if kind == "chunked":
        return ops.prefill_paged(s["q"], s["k_cache"], s["v_cache"], s["tables"], s["q_start"],
                                 s["q_len"], s["ctx"], s["longest"], k_scale=s["k_scale"],
                                 v_scale=s["v_scale"])
    if kind in ("prefill", "vision"):
        return ops.varlen_attention(s["q"], s["k"], s["v"], s["cu"], max_seqlen_q=s["longest"],
                                    causal=kind == "prefill")
    if kind == "rope":
        ops.qk_norm_rope_kv_write(s["q"], s["k"], s["v"], s["qw"], s["kw"], EPS, s["pos"],
                                  s["inv"], s["section"], s["k_cache"], s["v_cache"], s["slots"],
                                  s["k_scale"], s["v_scale"])
        out = dict(q=s["q"], k=s["k"], k_cache=s["k_cache"], v_cache=s["v_cache"])
        if s["k_scale"] is not None:
            out.update(k_scale=s["k_scale"], v_scale=s["v_scale"])
        return out
    md = s["md"]
    return dict(out=s["attn"](s["x"], s["pos"], metadata=md), k_cache=md.k_cache,
                v_cache=md.v_cache)


# ---- the work of a pass ------------------------------------------------------------------


def _es(case):
    """(bytes of a query / output element, bytes of a cached element with its scale's share)."""
    store = case.get("store", "bf16")
    return (4, 4) if store == "f32" else (2, 1 + 4 / D) if store == "fp8" else (2, 2)


def _chunk_pairs(prior, chunk):
    return chunk * prior + chunk * (chunk + 1) // 2


def work(case):
    kind = case["kind"]
    if kind == "vision":
        lens = _vision_lens(case)
        return {"bytes": 4 * sum(lens) * 16 * 80 * 2,
                "flops": 4 * 16 * 80 * sum(n * n for n in lens)}
    h, hkv = LAYOUTS[case["layout"]]
    es, ec = _es(case)
    if kind == "decode":
        lens = _lens(case)
        return {"bytes": sum(lens) * hkv * D * ec * 2 + 2 * len(lens) * h * D * es
                + 4 * sum(-(-n // case["block"]) for n in lens) + 8 * len(lens),
                "flops": 4 * h * D * sum(lens)}
    if kind == "prefill":
        lens = _lens(case)
        return {"bytes": sum(lens) * (2 * h + 2 * hkv) * D * es,
                "flops": 4 * h * D * sum(_chunk_pairs(0, n) for n in lens)}
    if kind == "chunked":
        c, prior = case["chunk"], _lens(case)
        return {"bytes": sum(n + c for n in prior) * hkv * D * ec * 2
                + 2 * len(prior) * c * h * D * es,
                "flops": 4 * h * D * sum(_chunk_pairs(n, c) for n in prior)}
    if kind == "rope":
        t = case["tokens"]
        return {"bytes": t * (2 * (h + hkv) + hkv) * D * es + 2 * t * hkv * D * ec
                + 8 * t * (4 if case["mrope"] else 2), "flops": 10 * t * (h + hkv) * D}
    dec, c, hidden = _lens(case), case["chunk"], HIDDEN[case["layout"]]
    t = len(dec) + c
    weights = hidden * (2 * h + 2 * hkv) * D
    return {"bytes": 2 * weights + 2 * 2 * t * hidden
            + (sum(dec) + case["prior"] + c) * hkv * D * 2 * 2,
            "flops": 2 * t * weights
            + 4 * h * D * (sum(dec) + _chunk_pairs(case["prior"], c))}


# ---- tolerances ----------------------------------------------------------------------------


def tolerance(case):
    kind, store = case["kind"], case.get("store", "bf16")
    if kind == "rope":
        if store == "f32":
            return {"rel": 1e-6, "max": 1e-5}
        # bf16 results on a rounding boundary move by one step (2^-8); fp8 codes likewise
        return {"rel": 2e-3, "max": 0.03, "differ": 0.01}
    if store == "f32":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": 1e-2, "max": 0.15}


# ---- the same in 64 bits -------------------------------------------------------------------


def _attend64(q, k, v, causal):
    """(L, H, D) x (S, H_kv, D): softmax attention, query row i seeing keys up to
    S - L + i when causal, in 64 bits."""
    n, h, d = q.shape
    s, hkv = k.shape[:2]
    out = torch.empty((n, h, d), dtype=torch.float64, device=q.device)
    g = h // hkv
    key = torch.arange(s, device=q.device)
    for j in range(hkv):
        kt, vj = k[:, j].double().t().contiguous(), v[:, j].double().contiguous()
        for i in range(0, n, 512):
            rows = q[i:i + 512, j * g:(j + 1) * g].double()
            x = rows.reshape(-1, d) @ kt / math.sqrt(d)
            if causal:
                last = torch.arange(i, i + rows.shape[0], device=q.device) + s - n
                hide = key[None, :] > last.repeat_interleave(g)[:, None]
                x.masked_fill_(hide, -math.inf)
            out[i:i + 512, j * g:(j + 1) * g] = (torch.softmax(x, -1) @ vj).view(rows.shape)
    return out


def _gather(s, cache, scale, i, n):
    """The first n cached rows of sequence i, (n, H_kv, D), in 64 bits."""
    rows = cache[s["tables"][i].long()]
    rows = rows.view(torch.float8_e4m3fn).double() * scale[s["tables"][i].long()].double()[
        ..., None] if scale is not None else rows.double()
    return rows.transpose(1, 2).reshape(-1, *rows.shape[1::2])[:n]


def _paged64(s, q, i, n):
    return _attend64(q, _gather(s, s["k_cache"], s["k_scale"], i, n),
                     _gather(s, s["v_cache"], s["v_scale"], i, n), True)


def _norm_rope64(x, w, pos, inv, section):
    """RMS norm (weight w or none) and rotary embedding; the angles are the fp32 products of
    position and frequency, as the models define them."""
    x = x.double()
    if w is not None:
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
    if section is not None:
        axis = torch.repeat_interleave(torch.arange(3), torch.tensor(section)).to(x.device)
        p = pos[axis].t()
    else:
        p = pos.unsqueeze(-1)
    ang = (p.float() * inv.float()).double().unsqueeze(1)
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat((a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()), -1)


def _write64(cache, rows, slots, block):
    """The cache in 64 bits with ``rows`` at their slots."""
    c = cache.double()
    c[slots // block, :, slots % block] = rows
    return c


def exact(case, seed):
    s = prepare(case, seed)
    kind = s["kind"]
    if kind in ("prefill", "vision"):
        cu = s["cu"].tolist()
        return torch.cat([_attend64(s["q"][a:b], s["k"][a:b], s["v"][a:b], kind == "prefill")
                          for a, b in zip(cu[:-1], cu[1:])])
    if kind in ("decode", "chunked"):
        c = case.get("chunk", 1)
        return torch.cat([_paged64(s, s["q"][i * c:(i + 1) * c], i, n)
                          for i, n in enumerate(s["ctx"].tolist())])
    if kind == "rope":
        q = _norm_rope64(s["q"], s["qw"], s["pos"], s["inv"], s["section"])
        k = _norm_rope64(s["k"], s["kw"], s["pos"], s["inv"], s["section"])
        if s["k_scale"] is None:
            return dict(q=q, k=k, k_cache=_write64(s["k_cache"], k, s["slots"], case["block"]),
                        v_cache=_write64(s["v_cache"], s["v"].double(), s["slots"],
                                         case["block"]))
        put = lambda sc, x: _write64(sc, x.abs().amax(-1) / 448, s["slots"],  # noqa: E731
                                     case["block"])
        return dict(q=q, k=k, k_cache=None, v_cache=None, k_scale=put(s["k_scale"], k),
                    v_scale=put(s["v_scale"], s["v"].double()))
    return _layer64(s, case)


def _layer64(s, case):
    attn, md, x, pos = s["attn"], s["md"], s["x"][0].double(), s["pos"][0]
    h, hkv = LAYOUTS[case["layout"]]
    lin = lambda m, n: (x @ m.weight.double().t()).view(-1, n, D)  # noqa: E731
    inv = attn.rotary.inv_freq
    q = _norm_rope64(lin(attn.q_proj, h), attn.q_norm.weight, pos, inv, None)
    k = _norm_rope64(lin(attn.k_proj, hkv), attn.k_norm.weight, pos, inv, None)
    slots = md.slot_mapping[0]
    kc = _write64(md.k_cache[0], k, slots, case["block"])
    vc = _write64(md.v_cache[0], lin(attn.v_proj, hkv), slots, case["block"])
    paged = dict(tables=md.kv_block_tables, k_cache=kc, v_cache=vc, k_scale=None, v_scale=None)
    out = torch.empty_like(q)
    for i, (a, n, c) in enumerate(zip(md.q_start.tolist(), md.q_len.tolist(),
                                      md.context_lens.tolist())):
        out[a:a + n] = _paged64(paged, q[a:a + n], i, c)
    out = out.reshape(out.shape[0], -1) @ attn.o_proj.weight.double().t()
    return dict(out=out.unsqueeze(0), k_cache=kc.unsqueeze(0), v_cache=vc.unsqueeze(0))
