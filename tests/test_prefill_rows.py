"""How the kernels divide their work, by the functions they run (csrc/work_map.h and
key_units.h, compiled for the host): every (sequence, head, row block) is some workgroup's
exactly once under each map, whatever remainder the groups and levels leave; the
multiply-shift division that splits packed rows into (token, head) agrees with the true one;
a DMA group of 16 packed rows stays within the span its buffer resource covers; ranges tile
the key tiles in order and none is empty; and few decode units take no more ranges than there
are, two to a range where that spares the merge a round."""
import ctypes
import itertools
import random

import pytest

from tests import work_map as wm


def cdiv(a, b):
    return -(-a // b)


def assert_covers(got, *axes):
    want = set(itertools.product(*axes))
    assert len(got) == len(want) and set(got) == want


@pytest.mark.parametrize("seqs,hkv,group", [(1, 1, 1), (3, 2, 4), (5, 4, 7), (9, 8, 2)])
@pytest.mark.parametrize("rows", [1, 128, 300, 400, 513, 1100])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("ranked", [False, True])
def test_maps_cover_the_work_once(seqs, hkv, group, rows, packed, ranked):
    g, n = wm.grid(seqs, hkv, group, rows, packed, ranked)
    order = random.Random(rows).sample(range(seqs), seqs)
    got = wm.mapped(g, "ranked" if ranked else "dense", n, order)
    heads = hkv if packed else hkv * group
    # no workgroup goes out for a level that no call has (an empty one costs what a short one does)
    assert n == 8 * cdiv(seqs * hkv, 8) * (heads // hkv) * cdiv(rows * g.pack, 128)
    assert_covers(got, range(seqs), range(heads), range(cdiv(rows * (group if packed else 1), 128)))


@pytest.mark.parametrize("seqs,hkv,group", [(3, 2, 4), (5, 4, 1), (9, 16, 1)])
def test_longest_levels_go_out_first(seqs, hkv, group):
    """Unpacked causal grids: a group's heads together, then the next shorter level of every
    group.  Runs of levels of one group are for packed heads only: with one head per KV head
    too they put long levels of the last groups behind short ones of the first."""
    g, n = wm.grid(seqs, hkv, group, 1100, False)
    levels = [m for _, _, m in wm.mapped(g, "dense", n)]
    assert levels == sorted(levels, reverse=True)


@pytest.mark.parametrize("seqs,hkv", [(1, 1), (3, 2), (9, 8), (17, 5)])
@pytest.mark.parametrize("blocks", [1, 3, 4, 5, 9])
def test_other_maps_cover_the_work_once(seqs, hkv, blocks):
    g = wm.Grid(num_seqs=seqs, num_kv_heads=hkv)
    for top_left, cut in itertools.product((0, 1), repeat=2):
        n = wm.lib().t_f32_grid(ctypes.byref(g), 64 * blocks - 3, top_left, cut)
        assert n == seqs * hkv * blocks  # every XCD takes its share, however few the groups
        got = [(s, h, m // 64) for s, h, m in wm.mapped(g, "f32", n)]
        assert_covers(got, range(seqs), range(hkv), range(blocks))
        if not top_left:  # a group's blocks together: they are equally long
            assert [x[:2] for x in got] == sorted(x[:2] for x in got)
    assert_covers(wm.mapped(g, "pair", 8 * cdiv(seqs, 8) * hkv), range(seqs), range(hkv), range(1))


def test_fp32_grid_takes_three_dimensions_past_one():
    """A dimension holds 2^24 - 1 workgroups of 256 threads."""
    for seqs, rows, run in ((1023, 131072, 4), (1024, 131072, 0), (65535, 1 << 20, 0),
                            (1, (1 << 31) - 1, 0), (8, (1 << 24) - 64 * 9, 4)):
        g = wm.Grid(num_seqs=seqs, num_kv_heads=8)
        n = wm.lib().t_f32_grid(ctypes.byref(g), rows, 1, 0)
        assert g.level_run == run and g.num_m_blocks == min(cdiv(rows, 64), (1 << 24) - 1)
        assert (n < 1 << 24) == (run > 0)


def test_division_by_the_group():
    div = wm.lib().t_div
    rng = random.Random(5)
    for d in list(range(2, 65)) + [80, 96, 100, 127, 128, 1000, 65535]:
        top = (1 << 31) - 1
        xs = set(range(200)) | {top, top - 1, top // d * d, top // d * d - 1}
        xs |= {b * 128 + o for b in (1, 7, 1023, 1 << 20) for o in (-1, 0, 1)}
        xs |= {rng.randrange(top // d) * d + o for o in (-1, 0, 1) for _ in range(50)}
        for x in xs:
            if 0 <= x <= top:
                assert div(x, d) == x // d, (x, d)


@pytest.mark.parametrize("qlen,group", [(1, 1), (40, 4), (33, 7), (129, 3), (128, 2), (5, 16)])
def test_packed_rows_stay_in_their_span(qlen, group):
    lib, q_tok, q_head, d = wm.lib(), 128 * 40, 128, 128
    tok = (lambda r: r) if group == 1 else (lambda r: lib.t_div(r, group))
    span = lib.t_span(q_tok, q_head, group, d)
    for g0 in range(0, qlen * group, 16):  # a DMA group of 16 rows, from its first row's token
        t0 = tok(g0)
        for r in range(g0, min(g0 + 16, qlen * group)):
            t = tok(r)
            assert 0 <= r - t * group < group
            assert 2 * ((t - t0) * q_tok + (r - t * group) * q_head + d) <= span


def test_ranges_tile_the_keys():
    lib = wm.lib()
    for tiles in list(range(0, 70)) + [127, 128, 129, 1000]:
        for splits, f32 in itertools.product((1, 2, 3, 5, 15, 31, 32), (0, 1)):
            n = lib.t_ranges(tiles, splits, f32)
            assert 1 <= n <= splits
            cut = [lib.t_range_tile(tiles, s, n) for s in range(n + 1)]
            assert cut[0] == 0 and cut[-1] == tiles
            least = 1 if f32 else 3
            assert n == 1 or all(b - a >= least for a, b in zip(cut, cut[1:]))
    for tiles in (4194305, (1 << 26) - 1, 1 << 26):  # 2^31 keys in tiles of 32
        for n in (32, 511, 512, 4096):
            assert [lib.t_range_tile(tiles, s, n) for s in (0, 1, n // 2, n - 1, n)] == \
                [tiles * s // n for s in (0, 1, n // 2, n - 1, n)]


@pytest.mark.parametrize("alone", [256, 1024, 17])
@pytest.mark.parametrize("resident", [1, 2])
@pytest.mark.parametrize("sequences", [1, 7, 130])
def test_few_decode_units_fit_the_ranges(alone, resident, sequences):
    lib = wm.lib()
    for total in {0, 1, 2, alone - 1, alone, alone + 1, 2 * alone - 1, 2 * alone}:
        assert lib.t_few(total, alone)
        per = lib.t_few_per(total, alone, resident * alone, sequences)
        assert cdiv(total, per) <= resident * alone
        # two units a range only where that spares the merge of a sequence a round
        assert (per == 2) == (total > alone and (resident == 1 or total > 16 * sequences))
    assert not lib.t_few(2 * alone + 1, alone)


def test_decode_merge_takes_more_waves_only_for_many_ranges_a_sequence():
    waves = wm.lib().t_merge_waves
    assert waves(16, 512, 2) == waves(256, 512, 32) == 16
    assert waves(28 * 36, 512, 36) == waves(32 * 32, 512, 2 * 32) == 4  # 14 and 8 ranges each
    assert waves(16 * 59, 512, 2 * 59) == waves(9 * 90, 2048, 3 * 90) == 1  # 4 and 7
    assert waves(32 * 64, 512, 64) == 1
