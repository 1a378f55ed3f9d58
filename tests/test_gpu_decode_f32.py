"""fp32 decode at 1e-5 (head_dim 128, block size 16, up to 8 query heads per KV head: every
group size, contexts on both sides of block, wave and partition edges, a block outside the
pool, and garbage past the context; head dims 64, 80 and 96 on both sides of their stage rule).
Oracle: oracle.textbook in float64."""
import pytest
import torch

from nano_inference_amd import ops, workloads
from tests.test_gpu_decode_shapes import oracle
from tests.tolerances import assert_attn_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g", range(1, 9))
def test_groups_and_edges(g):
    lens = [1, 15, 16, 17, 127, 128, 129, 144, 511, 512, 513, 1025, 1600]
    print(f"f32 decode G={g}", flush=True)
    c = workloads.make_decode(len(lens), 2 * g, 2, 128, lens, 400, 16, torch.float32, "cuda", 40 + g)
    for i, n in enumerate(lens):  # stale rows past the context, in its last block
        last = c.tables_list[i][-1]
        c.k_cache[0, last, :, (n - 1) % 16 + 1:] = float("nan")
        c.v_cache[0, last, :, (n - 1) % 16 + 1:] = float("inf")
    out = ops.paged_decode(c.q, c.k_cache[0], c.v_cache[0], c.block_tables, c.context_lens)
    assert_attn_close(out.double().cpu().numpy(), oracle(c), torch.float32)


@pytest.mark.parametrize("g", [1, 4, 5, 8])
@pytest.mark.parametrize("batch", [128, 129])
def test_many_sequences(batch, g):
    """Past 256 (sequence, KV head) pairs a workgroup has four waves instead of eight."""
    edges = [1, 16, 17, 63, 64, 65, 80, 129, 511, 512, 513, 1025]
    lens = [edges[i % len(edges)] for i in range(batch)]
    print(f"f32 decode G={g} batch={batch}", flush=True)
    c = workloads.make_decode(batch, 2 * g, 2, 128, lens, sum(-(-n // 16) for n in lens) + 5, 16,
                              torch.float32, "cuda", 60 + g)
    out = ops.paged_decode(c.q, c.k_cache[0], c.v_cache[0], c.block_tables, c.context_lens)
    assert_attn_close(out.double().cpu().numpy(), oracle(c), torch.float32)


@pytest.mark.parametrize("d", [64, 80, 96])
@pytest.mark.parametrize("batch,longest", [(16, 65), (17, 64), (17, 65), (3, 700), (128, 193), (129, 193)])
def test_stages_of_smaller_head_dims(d, batch, longest):
    """One LDS stage and two: tables of two tiles and of more, 64 workgroups and more, 512 and more."""
    edges = [1, 31, 32, 33, 63, 64, 65, 96, 97, 160, 193]
    lens = [longest] + [min(edges[i % len(edges)], longest) for i in range(batch - 1)]
    print(f"f32 decode D={d} batch={batch} longest={longest}", flush=True)
    c = workloads.make_decode(batch, 12, 4, d, lens, sum(-(-n // 16) for n in lens) + 5, 16,
                              torch.float32, "cuda", 70 + d)
    for i, n in enumerate(lens):
        last = c.tables_list[i][-1]
        c.k_cache[0, last, :, (n - 1) % 16 + 1:] = float("nan")
        c.v_cache[0, last, :, (n - 1) % 16 + 1:] = float("inf")
    out = ops.paged_decode(c.q, c.k_cache[0], c.v_cache[0], c.block_tables, c.context_lens)
    assert_attn_close(out.double().cpu().numpy(), oracle(c), torch.float32)


def test_block_outside_the_pool_is_skipped():
    c = workloads.make_decode(2, 8, 2, 128, [48, 700], 60, 16, torch.float32, "cuda", 39)
    whole = ops.paged_decode(c.q, c.k_cache[0], c.v_cache[0], c.block_tables, c.context_lens)
    c.block_tables[0, 2] = 1 << 20
    out = ops.paged_decode(c.q, c.k_cache[0], c.v_cache[0], c.block_tables, c.context_lens)
    assert torch.equal(out[1], whole[1])
    c.lens[0] = 32  # the same as a context that ends before it
    assert_attn_close(out.double().cpu().numpy(), oracle(c), torch.float32)
