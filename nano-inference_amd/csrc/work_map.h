// Which work a workgroup takes: the row blocks, grids and key ranges of the prefill kernels.
// Plain integer code for the device and for the host, as key_units.h.  The maps are templates
// over the kernels' parameter structs, whose fields they name.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "key_units.h"

template <typename T>
NIA_BOTH T at_least(T x, T lo) { return x > lo ? x : lo; }
template <typename T>
NIA_BOTH T at_most(T x, T hi) { return x < hi ? x : hi; }

// Workgroups of 256 threads along one dimension of a grid: HIP counts a dimension's threads in 32
// bits, refuses 2^32 and wraps beyond (a grid of 2^24 + 3 workgroups ran three of them).
constexpr int64_t kMaxGroups = ((int64_t)1 << 24) - 1;

// ---- bf16 prefill ------------------------------------------------------------------------------

constexpr int kBlockM = 128;  // query rows per workgroup
constexpr int kBlockN = 64;   // keys per tile
constexpr int kXcds = 8;
constexpr int kLevelRun = 4;

// Key tiles of an m-block of `tiles` tiles are cut into this many ranges (kSplitMinTiles each
// at least); range s takes tiles [tiles s / n, tiles (s + 1) / n).
constexpr int kSplitMinTiles = 4;
NIA_BOTH int key_ranges(int tiles, int splits) {
  return at_least(at_most(splits, tiles / kSplitMinTiles), 1);
}

// Workgroup -> (sequence, head, m-block) mapping of the 1-D prefill grid.
//
// The hardware hands workgroups to the 8 XCDs round-robin (id % 8), and each
// XCD has its own L2.  A (sequence, KV head) "group" owns the K/V rows that all
// its m-blocks and its G query heads read, so every group is pinned to one XCD
// (group % 8 == id % 8) and its K/V is fetched into one L2 only.  Inside an XCD
// the workgroups go out m-block-major from the bottom of the causal triangle,
// so the longest rows of every group start first and the short ones fill the
// tail.  Ids that map past the real work (uneven groups per XCD) return false.
// The grid holds no others: rounded up to whole runs of levels, three quarters of the packed
// grid of 100 prompts of 60 tokens (16 and 8 heads) were empty workgroups, about 10 ns each: 44
// us instead of 23, 300 of 20 tokens 94 instead of 29.
// The hardware hands an XCD's workgroups to its shader engines in turn, whatever each still
// has to do, so workgroups that follow each other must do about the same work: consecutive
// ones are the heads of one group and level, or where a KV head's heads are packed into the
// rows, kLevelRun adjacent levels of one group.  One level of every packed group in turn put
// each sequence on one engine: causal prefill of eight sequences of 256-4096 tokens 585 us
// instead of 320-335.  With one query head per KV head the levels go out in turn: in runs, 12
// prompts of up to 489 tokens (16 heads) took 26 us instead of 24, 40 of up to 180 (8 heads of
// 64) 12.7 instead of 8.7.
// RUNS: the grid may have packed heads (p.pack says whether it has).
template <bool RUNS, typename P>
NIA_BOTH bool prefill_map(const P& p, int id, int& seq, int& h, int& mb) {
  const int x = id % kXcds;
  const int t = id / kXcds;
  // `run` workgroups of one group follow each other: its heads of one level, or (packed heads)
  // kLevelRun levels of it, fewer where the levels end
  const bool heads = !RUNS || p.pack == 1;
  const int run = heads ? p.map_group : kLevelRun;
  const int per_z = p.groups_per_xcd * run;
  const int z0 = t / per_z;
  const int rem = t - z0 * per_z;
  const int len = heads ? run : at_most(run, p.num_m_blocks - z0 * run);
  const int j = rem / len;
  const int g = rem - j * len;
  const int gid = x + kXcds * j;
  const int z = heads ? z0 : z0 * kLevelRun + g;
  if (z >= p.num_m_blocks || gid >= p.num_seqs * p.num_kv_heads) return false;
  seq = gid / p.num_kv_heads;
  h = (gid - seq * p.num_kv_heads) * p.map_group + (heads ? g : 0);
  mb = p.num_m_blocks - 1 - z;
  return true;
}

// Paired-head grids (one query head per KV head, short unmasked sequences): all head pairs
// of a sequence on one XCD (sequence % 8), so the cache lines that two neighbouring pairs'
// rows share (a D = 80 row is 160 bytes) are fetched into one L2 once.
template <typename P>
NIA_BOTH bool pair_map(const P& p, int id, int& seq, int& h, int& mb) {
  const int x = id % kXcds;
  const int t = id / kXcds;
  const int j = t / p.num_kv_heads;
  seq = x + kXcds * j;
  h = t - j * p.num_kv_heads;
  mb = 0;
  return seq < p.num_seqs;
}

// Rank-major variant, for grids whose workgroups of one sequence all do about the same
// work (non-causal calls, and chunks after a cached context): sequences are ranked by
// key length (longest first), the groups of rank r go out before those of rank r + 1
// on every XCD (a group still lives on one XCD), and a group's m-blocks go out longest
// first.  Issuing the longest work first keeps a long sequence's workgroups out of the
// last round of the grid.  s_order[r] is the sequence of rank r.
template <typename P>
NIA_BOTH bool prefill_map_ranked(const P& p, int id, const int* s_order, int& seq, int& h,
                                 int& mb) {
  const int x = id % kXcds;
  const int t = id / kXcds;
  const int per_j = p.num_m_blocks * p.map_group;
  const int j = t / per_j;
  const int rem = t - j * per_j;
  const int z = rem / p.map_group;
  const int g = rem - z * p.map_group;
  const int gid = x + kXcds * j;
  if (j >= p.groups_per_xcd || gid >= p.num_seqs * p.num_kv_heads) return false;
  const int r = gid / p.num_kv_heads;
  seq = s_order[r];
  h = (gid - r * p.num_kv_heads) * p.map_group + g;
  mb = p.num_m_blocks - 1 - z;
  return true;
}

// Bytes that 16 consecutive packed rows of q span from the first one's token, head 0 of the
// group: at most 15 / pack + 1 tokens further (one token's rows may straddle two groups).
inline int64_t q_span_bytes(int64_t q_tok, int64_t q_head, int32_t pack, int head_dim) {
  const int64_t toks = pack == 1 ? 15 : 15 / pack + 1;
  return 2 * (toks * q_tok + (pack - 1) * q_head + head_dim);
}

// Key ranges per m-block for a grid of nwg workgroups whose m-blocks have at most `tiles` key
// tiles.  A lone workgroup takes about 1.1 us a tile, and the fp32 partials of a full chip's
// 512 workgroups about 13.6 us to write and read back, so n ranges cost 1.1 tiles / n +
// 13.6 n nwg / 512 us: least at n = sqrt(41 tiles / nwg).  At most what the chip holds at
// once (two workgroups a CU), and none where fewer than kSplitGain tiles are saved (the
// second launch).  Uncut, and in the ranges this takes (32 and 8 heads, one GPU): 64 rows after
// 8000 keys 146 us, 30 in 17; 24 rows after 16000 282, 26 in 32; eight 40-row chunks after
// 500-8192 keys 144, 64 in 4; 1024 rows after 12000 252, 222 in 2.  Top-left causal calls
// (`top_left`) stay uncut: their m-blocks average half the longest one's tiles, and a prompt of
// 2000 tokens (16 and 8 heads) in two ranges ran 42-44 us, uncut 38.
constexpr int kSplitSlots = 512;  // workgroups the chip holds at once
constexpr int kSplitMax = 32;
constexpr int kSplitGain = 12;

inline int32_t split_count(int64_t nwg, int64_t tiles, bool top_left) {
  if (top_left) return 1;
  int64_t n = kSplitSlots / nwg;
  if (n > kSplitMax) n = kSplitMax;
  if (n > tiles / kSplitMinTiles) n = tiles / kSplitMinTiles;
  while (n > 1 && n * n * nwg > 41 * tiles) --n;
  return n < 2 || tiles * (n - 1) < kSplitGain * n ? 1 : (int32_t)n;
}

inline size_t split_bytes(int64_t nwg, int32_t splits, int head_dim) {
  return splits > 1 ? (size_t)nwg * splits * kBlockM * ((size_t)head_dim + 2) * sizeof(float) : 0;
}

// Rows per item and m-blocks: the query heads of a KV head packed into the rows (p.pack =
// group), or one head an item.
template <typename P>
void set_rows(P& p, int max_q_len, bool packed) {
  p.pack = packed ? p.group : 1;
  p.map_group = packed ? 1 : p.group;
  p.num_m_blocks = (int32_t)(((int64_t)max_q_len * p.pack + kBlockM - 1) / kBlockM);
  block_divisor(p.pack, p.pack_magic, p.pack_shift);
}

// Blocks of 128 rows of a KV head's query heads: packed, and each head on its own.
inline int64_t packed_blocks(int32_t group, int max_q_len) {
  return ((int64_t)max_q_len * group + kBlockM - 1) / kBlockM;
}
inline int64_t head_blocks(int32_t group, int max_q_len) {
  return ((int64_t)max_q_len + kBlockM - 1) / kBlockM * group;
}

// Whether an uncut call packs: where the heads' own blocks need more than one round of the
// chip (two workgroups a CU) and packing saves a sixteenth of them.  Five prompts of 60-500
// tokens (28 and 4 heads) 22.6 -> 20.3 us, eight of 100-800 (16 and 8) 26.7 -> 24.8; with
// less to save, or a grid that fits the chip, the rows' divisions cost more than they bring
// (one prompt of 900 tokens 20.6 -> 21.1 us, six 60-row chunks 9.9 -> 10.7).  A call that is cut
// into key ranges packs whenever that saves a block: its blocks are what the ranges multiply.
template <typename P>
bool pack_uncut(const P& p, int max_q_len) {
  const int64_t own = head_blocks(p.group, max_q_len);
  return packed_blocks(p.group, max_q_len) * 16 <= own * 15 &&
         own * p.num_seqs * p.num_kv_heads > kSplitSlots;
}

// The workgroups of a packed or unpacked grid.
template <typename P>
int64_t grid_size(const P& p) {
  return (int64_t)kXcds * p.groups_per_xcd * p.map_group * p.num_m_blocks;
}

// ---- fp32 prefill ------------------------------------------------------------------------------

constexpr int kF32BlockM = 64;  // packed rows (query token, head of the group) per workgroup
constexpr int kF32BlockN = 32;  // keys per LDS tile

// Key ranges of about kF32RangeTiles tiles, so that no workgroup is left behind on a long row
// block (a tile takes 4.3 us and every workgroup's SIMDs are busy): four prompts of 128-1024
// tokens 217 us uncut, 183-186 in ranges of 5, 8 or 12 tiles; one of 500 77 us, 51 / 47 / 64.
// More than kF32SplitMaxRows rows (640 blocks) fill the chip evenly enough uncut: four prompts of
// 1000 tokens of 16 heads 281 us uncut, 314 in ranges; one 151 and 111.  The partials stay
// below kF32MaxParts x 33 KB (135 MB).
constexpr int kF32RangeTiles = 8;
constexpr int kF32SplitTiles = 12;   // fewer at most: uncut (the merge is a second launch)
constexpr int64_t kF32SplitMaxRows = 640 * kF32BlockM;  // NIA_PREFILL_F32_SPLIT_MAX_ROWS
constexpr int64_t kF32MaxParts = 4096;

NIA_BOTH int f32_ranges(int tiles, int splits) {
  return at_least(at_most(splits, (tiles + kF32RangeTiles - 1) / kF32RangeTiles), 1);
}

// Decode at a head dim below 128: two LDS stages where no CU has more than two workgroups, so
// that no third hides their loads (fp32, one stage and two): 32 sequences of 70 keys (16 heads of
// 96) 18.0 and 16.9 us, of 250 48.2 and 41.9, 76 of up to 827 (28 and 4 heads of 64) 101.7 and
// 86.5, 3 of 6032 601 and 572; 1016 workgroups of up to 786 keys (32 and 8 heads of 96) 234 and
// 250.  A context of two tiles gains nothing from the second stage (45 of up to 49, 6 and 2 heads
// of 96, 10.8 and 11.2), nor do 64 workgroups at a head dim of 80, which is no multiple of the
// four tiles a 16-byte read feeds (7 sequences of 2301 keys, 6 and 2 heads, 252.9 and 259.4; 112
// workgroups of 7920 keys 1154 and 1102).
constexpr int kF32PipeGroups = 512;
constexpr int kF32PipeKeys = 2 * kF32BlockN;
NIA_BOTH bool f32_two_stages(int head_dim, int64_t workgroups, int64_t table_keys) {
  return workgroups <= kF32PipeGroups && table_keys > kF32PipeKeys &&
         (head_dim != 80 || workgroups > 64);
}

// The workgroup's (sequence, KV head, row block).  `id`: its number in the 1-D grid, or x in a
// 3-D one (level_run 0) of row blocks, KV heads and sequences.  Runs of level_run adjacent
// levels of one (sequence, KV head) group follow each other (f32_run); the groups lie over all
// XCDs, since the matrix cores bound the tiles and not their loads: with every group on one
// XCD, four groups left half the chip idle (690 rows of 28 and 4 heads, D 96, 131 us instead of
// 73) and one XCD had the longest sequence to itself (seven of up to 775 rows of 8 heads and one
// 298 instead of 187); four prompts of 128-1024 tokens (16 and 8 heads) 186 and 182.
template <typename P>
NIA_BOTH void f32_map(const P& p, uint32_t id, uint32_t y, uint32_t z3, int& seq, int& hk,
                      int& m0) {
  int z;
  if (p.level_run == 0) {
    seq = (int)z3;
    hk = (int)y;
    z = (int)id;
  } else {
    const int per_level = p.groups * p.level_run;
    const int lv = (int)id / per_level;
    const int rem = (int)id - lv * per_level;
    const int len = at_most(p.level_run, p.num_m_blocks - lv * p.level_run);
    const int gid = rem / len;
    z = lv * p.level_run + (rem - gid * len);
    seq = gid / p.num_kv_heads;
    hk = gid - seq * p.num_kv_heads;
  }
  m0 = (p.num_m_blocks - 1 - z) * kF32BlockM;
}

// The row blocks of a call of at most `rows` packed rows a group, and all workgroups.  A sequence
// of more rows than a grid dimension holds blocks for would be a q of 2^30 rows.
inline int64_t f32_grid(int64_t groups, int64_t rows, int32_t& m_blocks) {
  m_blocks = (int32_t)at_most((rows + kF32BlockM - 1) / kF32BlockM, kMaxGroups);
  return groups * m_blocks;
}

// Adjacent levels of a group that follow each other in a grid of nwg workgroups; 0: the 3-D
// grid.  Top-left causal blocks are as long as their level: four levels of every group in turn,
// for the shader engines as in prefill_map.  Otherwise a group's blocks are about equally long
// and go out together, group by group, which the 3-D grid does without a division (ranges take
// its second dimension): with four levels in turn the last blocks of the longest image ended
// four images of 784-3072 rows (16 heads of 80) at 1528 us instead of 1293.  The 3-D grid is also
// for what one dimension does not hold (a loose row bound over very many sequences).
inline int32_t f32_run(int64_t nwg, int32_t m_blocks, bool top_left, bool cut) {
  if (!cut && (!top_left || nwg > kMaxGroups)) return 0;
  return top_left ? (m_blocks >= 4 ? 4 : 1) : m_blocks;
}

// `sure_rows`: query rows of the call as far as the launcher knows them (a single sequence's).
inline int32_t f32_split_count(int64_t nwg, int64_t max_k_len, int64_t sure_rows) {
  if (sure_rows > kF32SplitMaxRows) return 1;
  const int64_t tiles = (max_k_len + kF32BlockN - 1) / kF32BlockN;
  if (tiles < kF32SplitTiles) return 1;
  int64_t n = (tiles + kF32RangeTiles - 1) / kF32RangeTiles;
  if (n > kF32MaxParts / nwg) n = kF32MaxParts / nwg;
  return n < 2 ? 1 : (int32_t)n;
}

inline size_t f32_split_bytes(int64_t nwg, int32_t n, int head_dim) {
  return n > 1 ? (size_t)nwg * n * kF32BlockM * (sizeof(double) + (1 + head_dim) * sizeof(float)) : 0;
}

// ---- key tiles of a range (both kernels) ---------------------------------------------------------

// First tile of range s of n, floor(tiles s / n), for `tiles` tiles: the product itself does not
// fit an int (2^26 tiles of 32 keys in up to 512 ranges; n is at most kF32MaxParts).
NIA_BOTH int range_tile(int tiles, int s, int n) {
  const int q = tiles / n;
  return q * s + (tiles - q * n) * s / n;
}
