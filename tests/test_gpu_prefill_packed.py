"""Uncut prefill calls that pack a KV head's query heads into the row blocks: every row against
oracle.textbook in float64 (bars of tests.tolerances), for each mask, head dim, contiguous and
paged keys, rows that leave remainders in the 128-row blocks, and queries whose heads lie
apart.  That a case packs, and is not cut, is asked of the rule itself, so that a change of
its bounds fails here instead of leaving the packed kernels unrun."""
import math

import pytest
import torch

from nano_inference_amd import ops, workloads
from oracle import textbook as tb
from tests import work_map
from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu

CODES = {"top_left": ops.CAUSAL_TOP_LEFT, "none": ops.CAUSAL_NONE,
         "bottom_right": ops.CAUSAL_BOTTOM_RIGHT}
# (query heads, KV heads, D, query lengths, keys past the queries, mask)
CASES = [
    (32, 8, 128, [300, 17, 128, 129, 255, 1, 222, 300], 0, "top_left"),
    (28, 4, 128, [290, 18, 19, 37, 128, 183, 0, 289], 0, "top_left"),
    (16, 8, 80, [300, 1, 64, 127, 65, 299, 128, 2, 33, 200, 31], 0, "top_left"),
    (14, 2, 64, [100, 99, 1, 18, 19, 55] * 7, 0, "top_left"),
    (9, 3, 96, [170, 43, 42, 1, 128, 86] * 5, 0, "top_left"),
    (8, 2, 128, [40, 1, 31, 32, 33] * 60, 0, "top_left"),  # more than the ranking takes
    (32, 8, 128, [300, 17, 128, 129, 255, 1, 222, 300], 0, "none"),
    (28, 4, 80, [290, 18, 19, 37, 128, 183, 3, 289], 70, "bottom_right"),
    (32, 4, 96, [140, 16, 17, 8, 139, 128, 12, 100, 90, 80], 33, "bottom_right"),
]


def _check(h, hkv, d, n, longest, causal, rows):
    assert work_map.packs_uncut(n, hkv, h // hkv, longest)
    # the callers ask for ranges only up to this many rows
    assert causal == ops.CAUSAL_TOP_LEFT or n * h * longest > ops._SPLIT_MAX_ROWS or rows < 768


@pytest.mark.parametrize("layout", ["tokens", "heads"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_dense(case, layout):
    h, hkv, d, ql, more, mode = CASES[case]
    kl = [n + more * (i % 2) if n else 0 for i, n in enumerate(ql)]
    _check(h, hkv, d, len(ql), max(ql), CODES[mode], max(kl))
    print(f"packed {h}/{hkv} D {d} x{len(ql)} {mode} {layout}", flush=True)
    g = torch.Generator().manual_seed(400 + case)
    q, k, v = (torch.randn(s, generator=g).to(torch.bfloat16)
               for s in ((sum(ql), h, d), (sum(kl), hkv, d), (sum(kl), hkv, d)))
    qg = q.cuda() if layout == "tokens" else \
        q.transpose(0, 1).contiguous().cuda().transpose(0, 1)  # [H, T, D] memory
    starts = [torch.tensor([0] + x[:-1]).cumsum(0).to(torch.int32) for x in (ql, kl)]
    lens = [torch.tensor(x, dtype=torch.int32).cuda() for x in (ql, kl)]
    out = ops.prefill(qg, k.cuda(), v.cuda(), starts[0].cuda(), lens[0], starts[1].cuda(), lens[1],
                      max(ql), CODES[mode])
    o = out.double().cpu().numpy()
    res = tb.varlen(q.double().numpy(), k.double().numpy(), v.double().numpy(), starts[0].numpy(),
                    ql, starts[1].numpy(), kl, 1.0 / math.sqrt(d), mode)
    for s, (idx, ref) in res.items():
        if ql[s]:
            assert_attn_close(o[int(starts[0][s]) + idx], ref, torch.bfloat16, f"seq {s}")


# (query heads, KV heads, chunk, cached tokens before it, block size)
@pytest.mark.parametrize("h,hkv,chunk,prior,bs", [
    (32, 8, 300, [0, 500, 17, 64, 1, 200, 333, 90], 16),
    (28, 4, 290, [40, 0, 511, 128, 5, 64, 63, 250], 32), (16, 8, 161, [100, 3, 0, 64] * 5, 64)])
def test_paged(h, hkv, chunk, prior, bs):
    _check(h, hkv, 128, len(prior), chunk, ops.CAUSAL_BOTTOM_RIGHT, 1 << 30)
    print(f"packed paged {h}/{hkv} chunk {chunk} prior {prior} bs {bs}", flush=True)
    c = workloads.chunked_qwen3_8b("cuda", seed=410, n=len(prior), chunk=chunk, prior=prior,
                                   num_heads=h, num_kv_heads=hkv, block_size=bs)
    out = ops.prefill_paged(c.q, c.k_cache, c.v_cache, c.block_tables, c.q_start, c.q_len,
                            c.context_lens, c.chunk).double().cpu().numpy()
    res = tb.paged_prefill(c.q.double().cpu().numpy(), c.k_cache.double().cpu().numpy(),
                           c.v_cache.double().cpu().numpy(), c.block_tables.cpu().numpy(),
                           c.q_start.cpu().numpy(), c.q_len.cpu().numpy(),
                           c.context_lens.cpu().numpy(), 1.0 / math.sqrt(128))
    for s, (idx, ref) in res.items():
        assert_attn_close(out[s * chunk + idx], ref, torch.bfloat16, f"seq {s}")
