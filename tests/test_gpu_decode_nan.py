"""NaN through paged decode: a NaN query, NaN keys and a NaN value under a vanishing weight
poison their own output rows, whether one range holds the sequence or several are merged (by
one, four or sixteen waves a pair; fp32: one partition or several), and leave every other
output as it is without them."""
import pytest
import torch

from nano_inference_amd import ops, workloads
from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu

NAN = float("nan")

# (query heads, KV heads, contexts, block size): 16, 4 and 1 merging waves a pair, long rows in
# one range each (few units a sequence and many sequences), odd block sizes
CASES = [
    (16, 8, [2000, 31], 16), (16, 8, [1500] + [700] * 31, 16), (32, 8, [3000] + [900] * 39, 16),
    (32, 8, [200] * 300, 16), (28, 4, [40, 513], 16), (8, 2, [600, 100], 5),
]


def _unit(c, s):
    """(table block, row) of the 32 keys of a unit in the middle of sequence s, past no context."""
    j = c.lens[s] // 64
    return [(c.tables_list[s][t // c.block_size], t % c.block_size)
            for t in range(32 * j, min(32 * j + 32, c.lens[s]))]


def _output(c, store, what):
    """The decode's output with the NaNs of kind ``what`` in the first and the last sequence."""
    q, kc, vc, scales = c.q.clone(), c.k_cache[0].clone(), c.v_cache[0].clone(), {}
    if store == "fp8":
        f = workloads.quantize_cache_fp8(c)
        kc, vc = f.k_cache[0], f.v_cache[0]
        scales = dict(k_scale=f.k_scale[0].clone(), v_scale=f.v_scale[0].clone())
    for s in (0, len(c.lens) - 1):
        if what == "query":
            q[s, 1] = NAN
        for blk, row in _unit(c, s) if what == "keys" else _unit(c, s)[:1] if what == "value" else ():
            if store == "fp8":
                scales["k_scale" if what == "keys" else "v_scale"][blk, 1, row] = NAN
            elif what == "keys":
                kc[blk, 1, row] = NAN
            else:
                vc[blk, 1, row, 5] = NAN
    return ops.paged_decode(q, kc, vc, c.block_tables, c.context_lens, **scales).float().cpu()


@pytest.mark.parametrize("what", ["query", "keys", "value"])
@pytest.mark.parametrize("store", ["bf16", "fp8", "f32"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_nan(case, store, what):
    h, hkv, lens, bs = CASES[case]
    print(f"decode NaN {h}/{hkv} lens {lens[:3]} x{len(lens)} bs {bs} {store} {what}", flush=True)
    dtype = torch.float32 if store == "f32" else torch.bfloat16
    c = workloads.make_decode(len(lens), h, hkv, 128, lens, sum(-(-n // bs) for n in lens) + 2, bs,
                              dtype, "cuda", 51 + case)
    if what == "value":
        # the unit's keys point away from their head's queries: weights that underflow
        c.q[:, h // hkv:2 * (h // hkv), 0] = 40.0
        for s in (0, len(lens) - 1):
            for blk, row in _unit(c, s):
                c.k_cache[0, blk, 1, row] = 0
                c.k_cache[0, blk, 1, row, 0] = -400.0
    clean = _output(c, store, "")
    out = _output(c, store, what)
    group = slice(1, 2) if what == "query" else slice(h // hkv, 2 * (h // hkv))
    dims = slice(5, 6) if what == "value" and store != "fp8" else slice(None)
    bad = torch.zeros_like(out, dtype=torch.bool)
    for s in (0, len(lens) - 1):
        bad[s, group, dims] = True
    assert torch.isfinite(clean).all()
    assert torch.equal(torch.isnan(out), bad)
    # a NaN column leaves its running maximum, and with it the moments at which the others are
    # rescaled: they agree as two orders of one sum do (bars of tests.tolerances)
    assert_attn_close(out[~bad], clean[~bad], dtype)
