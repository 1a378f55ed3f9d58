"""The prefill grids and key ranges, as the kernels form them (CPU): every (sequence, head,
row block) is some workgroup's exactly once under each map, whatever remainder the groups
and levels leave; packed rows name each (token, head) once; ranges tile the key tiles in
order and none is empty; and the few-unit decode ranges hold every unit once."""
import itertools

import pytest

XCDS, BLOCK_M, LEVEL_RUN, MIN_TILES = 8, 128, 4, 4


def cdiv(a, b):
    return -(-a // b)


def dense_map(wg, seqs, hkv, map_group, m_blocks):
    """prefill_map: (sequence, head index, m-block) of workgroup wg, or None."""
    gpx = cdiv(seqs * hkv, XCDS)
    x, t = wg % XCDS, wg // XCDS
    heads = map_group > 1
    run = map_group if heads else LEVEL_RUN
    z0, rem = divmod(t, gpx * run)
    j, g = divmod(rem, run)
    gid, z = x + XCDS * j, z0 if heads else z0 * LEVEL_RUN + g
    if z >= m_blocks or gid >= seqs * hkv:
        return None
    seq = gid // hkv
    return seq, (gid - seq * hkv) * map_group + (g if heads else 0), m_blocks - 1 - z


def f32_map(wg, seqs, hkv, m_blocks):
    gpx, run = cdiv(seqs * hkv, XCDS), 4 if m_blocks >= 4 else 1
    x, wt = wg % XCDS, wg // XCDS
    lv, rem = divmod(wt, gpx * run)
    gj, r = divmod(rem, run)
    gid, z = x + XCDS * gj, lv * run + r
    if z >= m_blocks or gid >= seqs * hkv:
        return None
    return gid // hkv, gid % hkv, m_blocks - 1 - z


@pytest.mark.parametrize("seqs,hkv,group", [(1, 1, 1), (3, 2, 4), (5, 4, 7), (9, 8, 2)])
@pytest.mark.parametrize("m_blocks", [1, 3, 4, 5, 9])
def test_maps_cover_the_work_once(seqs, hkv, group, m_blocks):
    gpx = cdiv(seqs * hkv, XCDS)
    for map_group in {1, group}:
        levels = m_blocks if map_group > 1 else cdiv(m_blocks, LEVEL_RUN) * LEVEL_RUN
        got = [dense_map(w, seqs, hkv, map_group, m_blocks)
               for w in range(XCDS * gpx * map_group * levels)]
        got = [g for g in got if g is not None]
        want = set(itertools.product(range(seqs), range(hkv * map_group), range(m_blocks)))
        assert len(got) == len(want) and set(got) == want
    run = 4 if m_blocks >= 4 else 1
    got = [f32_map(w, seqs, hkv, m_blocks) for w in range(XCDS * gpx * cdiv(m_blocks, run) * run)]
    got = [g for g in got if g is not None]
    want = set(itertools.product(range(seqs), range(hkv), range(m_blocks)))
    assert len(got) == len(want) and set(got) == want


@pytest.mark.parametrize("qlen,group", [(1, 1), (40, 4), (33, 7), (129, 3), (128, 2), (5, 16)])
def test_packed_rows_and_their_span(qlen, group):
    rows = [(r // group, r % group) for r in range(qlen * group)]
    assert len(set(rows)) == qlen * group
    toks = 15 if group == 1 else 15 // group + 1  # q_span_bytes
    for g0 in range(0, qlen * group, 16):  # a DMA group of 16 rows
        t0 = rows[g0][0]
        assert max(t for t, _ in rows[g0:g0 + 16]) - t0 <= toks


def test_ranges_tile_the_keys():
    for tiles in list(range(0, 70)) + [127, 128, 129, 1000]:
        for splits in (1, 2, 3, 5, 15, 31, 32):
            n = max(1, min(splits, tiles // MIN_TILES))
            cut = [tiles * s // n for s in range(n + 1)]
            assert cut[0] == 0 and cut[-1] == tiles
            assert n == 1 or all(b - a >= MIN_TILES - 1 and b > a for a, b in zip(cut, cut[1:]))
            n = max(1, min(splits, cdiv(tiles, 8)))  # the fp32 kernel's
            cut = [tiles * s // n for s in range(n + 1)]
            assert cut[-1] == tiles and (tiles == 0 or all(b > a for a, b in zip(cut, cut[1:])))


@pytest.mark.parametrize("alone,grid_waves", [(256, 512), (1024, 2048), (17, 40)])
def test_few_decode_units_lie_in_one_range_each(alone, grid_waves):
    for total in {1, 2, alone - 1, alone, alone + 1, 2 * alone - 1, 2 * alone}:
        per = 1 if total <= alone else 2
        ranges = [(min(v * per, total), min(v * per + per, total)) for v in range(grid_waves)]
        units = [u for a, b in ranges for u in range(a, b)]
        assert units == list(range(total))
        assert sum(a < b for a, b in ranges) == cdiv(total, per) <= alone
