"""Prefill calls with few query rows: the query heads of a KV head packed into one row block,
and row blocks whose keys are cut into ranges and merged (nia_prefill_split,
nia_prefill_paged_split, and over fp8 caches).  Row counts around a block's remainder, key
counts around range and tile edges, one call holding both cut and uncut sequences, rows and
ranges that see no key, layouts whose query heads lie far apart, and the call without a
workspace.  Oracle: oracle.textbook in float64; bars of tests.tolerances."""
import math

import numpy as np
import pytest
import torch

from nano_inference_amd import _lib, ops, workloads
from oracle import fp8_kv as F
from oracle import textbook as tb
from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu


def _randn(shape, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g).to(torch.bfloat16)


# (query heads, KV heads, chunk, cached tokens before it, block size)
PAGED = [
    (4, 1, 1, [4096, 0, 63, 1000], 16), (32, 8, 24, [3000], 16), (7, 1, 40, [2500, 130], 32),
    (28, 4, 33, [1500, 1, 767], 16), (2, 2, 129, [1311], 64), (16, 8, 300, [1000], 16),
    (8, 2, 17, [5000 + 47, 5000 + 48], 16), (32, 2, 5, [64 * 48 - 5, 64 * 48 - 4], 16),
    (3, 1, 43, [900, 1999], 16), (8, 8, 128, [2000], 16), (5, 1, 200, [12, 3], 16),
]


@pytest.mark.parametrize("store", ["bf16", "fp8"])
@pytest.mark.parametrize("case", range(len(PAGED)))
def test_paged(case, store):
    h, hkv, chunk, prior, bs = PAGED[case]
    print(f"ranges paged {h}/{hkv} chunk {chunk} prior {prior} bs {bs} {store}", flush=True)
    c = workloads.chunked_qwen3_8b("cuda", seed=70 + case, n=len(prior), chunk=chunk, prior=prior,
                                   num_heads=h, num_kv_heads=hkv, block_size=bs)
    caches, scales = (c.k_cache, c.v_cache), (None, None)
    exp_k, exp_v = (x.double().cpu().numpy() for x in caches)
    if store == "fp8":
        pairs = [F.quantize_rows(x.cpu()) for x in caches]
        exp_k, exp_v = (F.dequantize_rows(q, s).double().numpy() for q, s in pairs)
        caches, scales = [q.cuda() for q, _ in pairs], [s.contiguous().cuda() for _, s in pairs]
    out = ops.prefill_paged(c.q, *caches, c.block_tables, c.q_start, c.q_len, c.context_lens,
                            c.chunk, k_scale=scales[0], v_scale=scales[1])
    o = out.double().cpu().numpy()
    res = tb.paged_prefill(c.q.double().cpu().numpy(), exp_k, exp_v, c.block_tables.cpu().numpy(),
                           c.q_start.cpu().numpy(), c.q_len.cpu().numpy(),
                           c.context_lens.cpu().numpy(), 1.0 / math.sqrt(128))
    for s, (idx, ref) in res.items():
        assert_attn_close(o[s * chunk + idx], ref, torch.bfloat16, f"seq {s}")


# (query heads, KV heads, D, query lengths, key lengths, mode)
DENSE = [
    (4, 1, 128, [10, 200], [3000, 900], "bottom_right"), (2, 1, 64, [7], [1600], "none"),
    (4, 4, 80, [100, 1], [2100, 1], "none"), (6, 2, 96, [50], [1537], "none"),
    (4, 2, 128, [1200, 3], [1000, 2000], "bottom_right"),  # rows that see no key
    (8, 1, 128, [33], [1024], "none"), (7, 1, 128, [20, 300, 5], [20, 300, 5], "top_left"),
    (3, 1, 80, [45, 43], [45, 43], "top_left"), (2, 2, 128, [77, 700], [77, 700], "top_left"),
]


@pytest.mark.parametrize("layout", ["tokens", "heads", "far"])
@pytest.mark.parametrize("case", range(len(DENSE)))
def test_dense(case, layout):
    h, hkv, d, ql, kl, mode = DENSE[case]
    print(f"ranges dense {h}/{hkv} D {d} q {ql} k {kl} {mode} {layout}", flush=True)
    tq, tk = sum(ql), sum(kl)
    q, k, v = (_randn(s, 300 + case) for s in ((tq, h, d), (tk, hkv, d), (tk, hkv, d)))
    if layout == "tokens":
        qg = q.cuda()
    else:  # heads apart: [H, T, D], or farther than packed rows can reach
        step = tq * d if layout == "heads" else 1 << 26
        buf = torch.empty((h - 1) * step + tq * d, dtype=torch.bfloat16, device="cuda")
        qg = buf.as_strided((tq, h, d), (d, step, 1))
        qg.copy_(q)
    starts = [torch.tensor([0] + x[:-1]).cumsum(0).to(torch.int32).cuda() for x in (ql, kl)]
    lens = [torch.tensor(x, dtype=torch.int32).cuda() for x in (ql, kl)]
    code = {"top_left": ops.CAUSAL_TOP_LEFT, "none": ops.CAUSAL_NONE,
            "bottom_right": ops.CAUSAL_BOTTOM_RIGHT}[mode]
    out = ops.prefill(qg, k.cuda(), v.cuda(), starts[0], lens[0], starts[1], lens[1], max(ql), code)
    o = out.double().cpu().numpy()
    res = tb.varlen(q.double().numpy(), k.double().numpy(), v.double().numpy(),
                    starts[0].cpu().numpy(), ql, starts[1].cpu().numpy(), kl,
                    1.0 / math.sqrt(d), mode)
    for s, (idx, ref) in res.items():
        at = int(starts[0][s])
        assert_attn_close(o[at + idx], ref, torch.bfloat16, f"seq {s}")


def test_large_logits_across_ranges():
    """A key that dominates its row lies in one range; the others' weights underflow there."""
    c = workloads.chunked_qwen3_8b("cuda", seed=99, n=1, chunk=16, prior=[4000], num_heads=8,
                                   num_kv_heads=2)
    c.k_cache *= 6
    out = ops.prefill_paged(c.q, c.k_cache, c.v_cache, c.block_tables, c.q_start, c.q_len,
                            c.context_lens, c.chunk).double().cpu().numpy()
    res = tb.paged_prefill(c.q.double().cpu().numpy(), c.k_cache.double().cpu().numpy(),
                           c.v_cache.double().cpu().numpy(), c.block_tables.cpu().numpy(),
                           c.q_start.cpu().numpy(), c.q_len.cpu().numpy(),
                           c.context_lens.cpu().numpy(), 1.0 / math.sqrt(128))
    assert_attn_close(out[res[0][0]], res[0][1], torch.bfloat16)


def test_workspace_decides_and_never_fails():
    """Without a workspace, or with one too small, the call runs uncut."""
    c = workloads.chunked_qwen3_8b("cuda", seed=98, n=2, chunk=24, prior=[3000, 40], num_heads=8,
                                   num_kv_heads=2)
    lib = _lib.load()
    mb = c.block_tables.shape[1]
    need = lib.nia_prefill_split_workspace_size(2, 24, mb * 16, 8, 2, 128,
                                                ops.CAUSAL_BOTTOM_RIGHT, 0)
    assert need > 0
    outs = []
    for nbytes in (0, need - 1, need):
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        out = torch.empty_like(c.q)
        st = lib.nia_prefill_paged_split(
            out.data_ptr(), out.stride(0), out.stride(1), c.q.data_ptr(), c.q.stride(0),
            c.q.stride(1), c.k_cache.data_ptr(), c.v_cache.data_ptr(), c.block_tables.data_ptr(),
            mb, mb, c.q_start.data_ptr(), c.q_len.data_ptr(), c.context_lens.data_ptr(), 2, 24, 8,
            2, 128, 16, c.k_cache.shape[0], 1.0 / math.sqrt(128), ops.CAUSAL_BOTTOM_RIGHT, 0,
            ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream)
        assert st == _lib.OK
        outs.append(out.float().cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    assert np.abs(outs[2] - outs[0]).max() <= 2e-2
    assert np.array_equal(outs[2][24:], outs[0][24:])  # the short sequence is never cut


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_nan_and_infinity_come_through_the_merge(dtype):
    """A NaN query, a NaN value under a vanishing weight and an infinite key poison the rows
    that an uncut call (no workspace) poisons, and no others."""
    c = workloads.chunked_qwen3_8b("cuda", dtype=dtype, seed=96, n=1, chunk=24, prior=[3000],
                                   num_heads=8, num_kv_heads=2)
    c.q[3, 1] = float("nan")
    c.q[:, 4:] *= 40  # the second KV head's group: weights that underflow
    c.v_cache[c.tables_list[0][2], 1, 3, 5] = float("nan")
    c.k_cache[c.tables_list[0][100], 0, 0] = float("inf")
    lib, mb = _lib.load(), c.block_tables.shape[1]
    code = ops._DTYPES[dtype]
    need = lib.nia_prefill_split_workspace_size(1, 24, mb * 16, 8, 2, 128, ops.CAUSAL_BOTTOM_RIGHT,
                                                code)
    assert need > 0
    ws, outs = torch.empty(need, dtype=torch.uint8, device="cuda"), []
    for nbytes in (0, need):
        out = torch.empty_like(c.q)
        st = lib.nia_prefill_paged_split(
            out.data_ptr(), out.stride(0), out.stride(1), c.q.data_ptr(), c.q.stride(0),
            c.q.stride(1), c.k_cache.data_ptr(), c.v_cache.data_ptr(), c.block_tables.data_ptr(),
            mb, mb, c.q_start.data_ptr(), c.q_len.data_ptr(), c.context_lens.data_ptr(), 1, 24, 8,
            2, 128, 16, c.k_cache.shape[0], 1.0 / math.sqrt(128), ops.CAUSAL_BOTTOM_RIGHT, code,
            ws.data_ptr() if nbytes else None, nbytes, torch.cuda.current_stream().cuda_stream)
        assert st == _lib.OK
        outs.append(out.float().cpu())
    assert torch.isnan(outs[0][3, 1]).all() and torch.isnan(outs[0][:, 4:, 5]).any()
    assert torch.equal(torch.isnan(outs[0]), torch.isnan(outs[1]))


def test_captured_call_replays():
    """A cut call under HIP graph capture, replayed with eager calls in between."""
    c = workloads.chunked_qwen3_8b("cuda", seed=97, n=1, chunk=24, prior=[3000], num_heads=8,
                                   num_kv_heads=2)
    args = (c.q, c.k_cache, c.v_cache, c.block_tables, c.q_start, c.q_len, c.context_lens, c.chunk)
    eager = ops.prefill_paged(*args)
    torch.cuda.synchronize()
    graph, out = torch.cuda.CUDAGraph(), torch.empty_like(c.q)
    with torch.cuda.graph(graph):
        ops.prefill_paged(*args, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert torch.equal(ops.prefill_paged(*args), eager)


@pytest.mark.parametrize("dtype,ql,kl,cut", [
    (torch.bfloat16, [32] * 16, [700] * 16, False), (torch.bfloat16, [64], [8000], True),
    (torch.bfloat16, [1] * 3, [2235, 560, 1300], True),
    (torch.float32, [8] * 20, [100] * 20, False), (torch.float32, [200], [900], True),
    (torch.float32, [30, 400, 10], [30, 400, 10], True), (torch.float32, [30] * 14, [30] * 14, False)])
def test_ranges_are_chosen_for_one_sequence_not_for_the_sum(monkeypatch, dtype, ql, kl, cut):
    """Many short sequences are not cut for the sum of their keys."""
    seen, ask = [], ops._split_workspace
    monkeypatch.setattr(ops, "_split_workspace", lambda *a: seen.append(ask(*a)) or seen[-1])
    h, hkv, d = 16, 8, 128
    q, k, v = (_randn((sum(n), m, d), 5).to(dtype).cuda() for n, m in ((ql, h), (kl, hkv), (kl, hkv)))
    starts = [torch.tensor([0] + x[:-1]).cumsum(0).to(torch.int32).cuda() for x in (ql, kl)]
    lens = [torch.tensor(x, dtype=torch.int32).cuda() for x in (ql, kl)]
    ops.prefill(q, k, v, starts[0], lens[0], starts[1], lens[1], max(ql), ops.CAUSAL_NONE)
    assert any(x is not None for x in seen) == cut


@pytest.mark.parametrize("bs,cut", [(16, True), (64, True), (24, False), (12, False), (5, False)])
def test_block_sizes_that_are_never_cut_ask_for_no_workspace(monkeypatch, bs, cut):
    seen, ask = [], ops._split_workspace
    monkeypatch.setattr(ops, "_split_workspace", lambda *a: seen.append(ask(*a)) or seen[-1])
    c = workloads.chunked_qwen3_8b("cuda", seed=95, n=1, chunk=24, prior=[3000], num_heads=8,
                                   num_kv_heads=2, block_size=bs)
    ops.prefill_paged(c.q, c.k_cache, c.v_cache, c.block_tables, c.q_start, c.q_len,
                      c.context_lens, c.chunk)
    assert any(x is not None for x in seen) == cut
