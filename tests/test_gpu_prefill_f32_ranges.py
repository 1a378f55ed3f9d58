"""The fp32 prefill kernel's row and range forms at 1e-5: query heads packed into the row
blocks of 64, key ranges and their merge (dense and paged), tile and range edges, rows and
ranges that see no key, an additive mask, and head dims whose output tiles do not come in
fours.  Oracle: oracle.textbook in float64."""
import math

import pytest
import torch

from nano_inference_amd import ops, workloads
from oracle import textbook as tb
from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu

# (query heads, KV heads, D, query lengths, key lengths, mode)
DENSE = [
    (2, 1, 128, [400, 3, 383], [400, 3, 383], "top_left"), (7, 1, 64, [37], [900], "none"),
    (4, 4, 80, [65, 1], [385, 32], "none"), (6, 2, 96, [50], [417], "bottom_right"),
    (4, 2, 128, [600, 3], [500, 700], "bottom_right"), (3, 1, 128, [21, 22], [21, 22], "top_left"),
    (8, 1, 128, [8], [1024 + 31], "none"), (16, 8, 128, [385], [385], "top_left"),
]


@pytest.mark.parametrize("case", range(len(DENSE)))
def test_dense(case):
    h, hkv, d, ql, kl, mode = DENSE[case]
    print(f"f32 ranges dense {h}/{hkv} D {d} q {ql} k {kl} {mode}", flush=True)
    g = torch.Generator().manual_seed(500 + case)
    q, k, v = (torch.randn(s, generator=g)
               for s in ((sum(ql), h, d), (sum(kl), hkv, d), (sum(kl), hkv, d)))
    starts = [torch.tensor([0] + x[:-1]).cumsum(0).to(torch.int32).cuda() for x in (ql, kl)]
    lens = [torch.tensor(x, dtype=torch.int32).cuda() for x in (ql, kl)]
    code = {"top_left": ops.CAUSAL_TOP_LEFT, "none": ops.CAUSAL_NONE,
            "bottom_right": ops.CAUSAL_BOTTOM_RIGHT}[mode]
    out = ops.prefill(q.cuda(), k.cuda(), v.cuda(), starts[0], lens[0], starts[1], lens[1],
                      max(ql), code)
    o = out.double().cpu().numpy()
    res = tb.varlen(q.double().numpy(), k.double().numpy(), v.double().numpy(),
                    starts[0].cpu().numpy(), ql, starts[1].cpu().numpy(), kl,
                    1.0 / math.sqrt(d), mode)
    for s, (idx, ref) in res.items():
        assert_attn_close(o[int(starts[0][s]) + idx], ref, torch.float32, f"seq {s}")


@pytest.mark.parametrize("h,hkv,chunk,prior,bs", [
    (4, 1, 1, [700, 0], 16), (16, 8, 33, [351, 352], 5), (7, 1, 20, [1500], 32), (2, 2, 70, [400], 1)])
def test_paged(h, hkv, chunk, prior, bs):
    print(f"f32 ranges paged {h}/{hkv} chunk {chunk} prior {prior} bs {bs}", flush=True)
    c = workloads.chunked_qwen3_8b("cuda", dtype=torch.float32, seed=60, n=len(prior), chunk=chunk,
                                   prior=prior, num_heads=h, num_kv_heads=hkv, block_size=bs)
    out = ops.prefill_paged(c.q, c.k_cache, c.v_cache, c.block_tables, c.q_start, c.q_len,
                            c.context_lens, c.chunk).double().cpu().numpy()
    res = tb.paged_prefill(c.q.double().cpu().numpy(), c.k_cache.double().cpu().numpy(),
                           c.v_cache.double().cpu().numpy(), c.block_tables.cpu().numpy(),
                           c.q_start.cpu().numpy(), c.q_len.cpu().numpy(),
                           c.context_lens.cpu().numpy(), 1.0 / math.sqrt(128))
    for s, (idx, ref) in res.items():
        assert_attn_close(out[s * chunk + idx], ref, torch.float32, f"seq {s}")


def test_additive_mask_over_packed_heads():
    b, h, hkv, s, d = 2, 6, 2, 70, 128
    g = torch.Generator().manual_seed(61)
    q = torch.randn(b * s, h, d, generator=g)
    k, v = (torch.randn(b * s, hkv, d, generator=g) for _ in range(2))
    mask = torch.randn(b, h, s, s, generator=g)
    mask[torch.rand(mask.shape, generator=g) < 0.2] = -math.inf
    at, n = torch.arange(b, dtype=torch.int32).cuda() * s, torch.full((b,), s, dtype=torch.int32).cuda()
    out = ops.prefill(q.cuda(), k.cuda(), v.cuda(), at, n, at, n, s, ops.CAUSAL_NONE,
                      mask=mask.cuda()).double().cpu()
    qd, kd, vd = (x.double().view(b, s, -1, d).transpose(1, 2) for x in (q, k, v))
    kd, vd = (x.repeat_interleave(h // hkv, 1) for x in (kd, vd))
    ref = torch.softmax(qd @ kd.transpose(2, 3) / math.sqrt(d) + mask.double(), -1) @ vd
    assert_attn_close(out.numpy(), ref.transpose(1, 2).reshape(b * s, h, d).numpy(), torch.float32)


@pytest.mark.parametrize("paged", [False, True])
def test_many_sequences_under_a_loose_row_bound(paged):
    """2^24 row blocks of 256 threads: one grid dimension does not hold them."""
    n, h, d, bound = 1024, 8, 64, 131072
    g = torch.Generator().manual_seed(62)
    ql = [1 + i % 3 if i % 100 == 7 else 0 for i in range(n)]
    ql[n - 1] = 2
    q, k, v = (torch.randn(sum(ql), h, d, generator=g) for _ in range(3))
    at = torch.tensor([0] + ql[:-1]).cumsum(0).to(torch.int32)
    lens = torch.tensor(ql, dtype=torch.int32)
    if paged:
        tables = torch.zeros(n, 1, dtype=torch.int32)
        used = [s for s in range(n) if ql[s]]
        cache = torch.zeros(2, len(used), h, 4, d)
        for b, s in enumerate(used):
            tables[s] = b
            for i, x in enumerate((k, v)):
                cache[i, b, :, :ql[s]] = x[at[s]:at[s] + ql[s]].transpose(0, 1)
        kc, vc = cache.cuda()
        out = ops.prefill_paged(q.cuda(), kc, vc, tables.cuda(), at.cuda(), lens.cuda(),
                                lens.to(torch.int64).cuda(), bound, ops.CAUSAL_BOTTOM_RIGHT)
    else:
        out = ops.prefill(q.cuda(), k.cuda(), v.cuda(), at.cuda(), lens.cuda(), at.cuda(),
                          lens.cuda(), bound, ops.CAUSAL_TOP_LEFT)
    o = out.double().cpu().numpy()
    res = tb.varlen(q.double().numpy(), k.double().numpy(), v.double().numpy(), at.numpy(), ql,
                    at.numpy(), ql, 1.0 / math.sqrt(d), "top_left")
    for s, (idx, ref) in res.items():
        if ql[s]:
            assert_attn_close(o[int(at[s]) + idx], ref, torch.float32, f"seq {s}")
