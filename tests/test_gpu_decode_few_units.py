"""Decodes of few units (one or two per range) and of sequences cut into many ranges, whose
merge takes one, four or sixteen waves per (sequence, head): unit totals on both sides of
the ranges' one-unit and two-unit limits, and sequences of 16 / 17, 64 / 65 and 256 / 257
ranges.  Oracle and bars as in test_gpu_decode_shapes."""
import pytest
import torch

from nano_inference_amd import ops, workloads
from tests.test_gpu_decode_shapes import oracle, step
from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu

U = 32  # keys per unit

# (query heads, KV heads, contexts).  256 CUs: one unit a range up to 256 units times the
# slices per KV head (4 / KV heads per workgroup), two up to twice that, weighted beyond.
CASES = [
    (16, 8, [1]), (16, 8, [16 * U, 17 * U, 0, 5]), (32, 8, [64 * U, 63 * U + 1]),
    (16, 8, [65 * U]), (4, 4, [256 * U - 1]), (4, 4, [257 * U]), (4, 4, [512 * U]),
    (4, 4, [513 * U]), (8, 1, [1024 * U - 3]), (8, 1, [1025 * U]), (2, 2, [300 * U, 0, 2000]),
    (28, 4, [40 * U] * 10), (28, 4, [17 * U] * 36), (32, 8, [40 * U + 1] * 33),
]


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_few_units(case, fp8):
    h, hkv, lens = CASES[case]
    print(f"few units {h}/{hkv} lens {lens[:4]} x{len(lens)} fp8={fp8}", flush=True)
    blocks = sum(-(-n // 16) for n in lens)
    # an empty sequence still writes its new token, into a block of its own
    drawn = [max(n, 1) for n in lens]
    c = workloads.make_decode(len(lens), h, hkv, 128, drawn, blocks + len(lens) + 3, 16,
                              torch.bfloat16, "cuda", 91 + case)
    c.lens = list(lens)
    c.context_lens = torch.tensor(lens, dtype=torch.int64, device="cuda")
    if not fp8:
        out = step(c)
        assert_attn_close(out.double().cpu().numpy(), oracle(c), torch.bfloat16)
        return
    f = workloads.quantize_cache_fp8(c)
    out = ops.paged_decode(c.q, f.k_cache[0], f.v_cache[0], c.block_tables, c.context_lens,
                           k_scale=f.k_scale[0], v_scale=f.v_scale[0])
    c.k_cache, c.v_cache = (x.double() for x in (c.k_cache, c.v_cache))
    for cache, codes, scale in ((c.k_cache, f.k_cache, f.k_scale), (c.v_cache, f.v_cache, f.v_scale)):
        cache.copy_(codes.view(torch.float8_e4m3fn).double() * scale.unsqueeze(-1).double())
    assert_attn_close(out.double().cpu().numpy(), oracle(c), torch.bfloat16)
