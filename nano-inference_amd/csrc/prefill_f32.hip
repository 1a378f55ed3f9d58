// fp32 varlen prefill attention (causal / non-causal, contiguous or paged K/V) for gfx950.
//
// The fp32 mode of the reference's attention (its shipped configs run float32,
// configs/default.yaml:4): the prefill branch of src/nano_inference/layers/attention.py:
// 281-284 with scaled_dot_product_attention (:12-50), the vision tower's per-chunk loop
// (src/nano_inference/layers/vision.py:190-208), and chunked prefill over the paged cache.
// Same varlen description and causal modes as the bf16 kernels (include/nia_attn.h).
// The same kernel reads bf16 and fp8 paged caches whose block size the bf16 / fp8 kernels
// do not take (they find a key's block with a shift; the reference's block size is any
// positive integer, src/nano_inference/core/config.py:54): decode (one query row per
// sequence, src/nano_inference/layers/attention.py:285-332) and bf16 chunked prefill.
//
// Precision: every score q . k is summed on the fp64 matrix cores
// (v_mfma_f64_16x16x4_f64, fp32 inputs widened exactly), so it carries no accumulated
// rounding even at logits of ~100 nats, where an fp32 sum of 128 products is already
// ~1e-5 off; the softmax keeps its running max in fp64 and its weights, sums and the
// output in fp32 (P V on v_mfma_f32_16x16x4_f32).
//
// Bound by the matrix cores: per (query, key) 2 D FLOP in fp64 (78.6 TFLOP/s on this chip)
// and 2 D in fp32 (157), 4096 + 2048 cycles of a SIMD for a wave's 16 x 32 tile at D = 128.
// Tiling: a workgroup of 4 waves owns 64 packed rows (16 per wave): row r is query token
// r / G, head r % G of a KV head's G query heads, so the heads of a group share their K/V
// tiles and a decode's G heads fill one wave's columns.  Key tiles of 32 rows are staged in LDS
// (fp32, 16-byte chunks permuted within a row: swz).  D 128, whose registers leave two
// workgroups a CU: a tile is loaded into registers while the one before is computed on, and
// written to the other of two stages; operands are read from LDS a step ahead.  Smaller D: one
// stage and no read-ahead, which leaves room for three workgroups a CU (D 64: four) that hide
// each other's loads: four images of 784-3072 rows (16 heads of 80) 1633 us with two stages and
// two workgroups, 1528 so, 114 windows of 16-64 rows 61.5 and 52.0 (54 with 512-byte rows left
// out but two stages kept), 109 decodes of up to 40 keys (16 heads of 64) 27.7 and 18.1.  Decodes
// of at most two workgroups a CU keep two stages (f32_two_stages).
// Against one head a block, tiles loaded behind a barrier each and the shortest blocks
// first: four prompts of 128-1024 tokens (16 and 8 heads, D 128) 268 -> 182 us, one of 1000
// 192 -> 111, four of 1000 551 -> 281.  The fp64 products bound it: v_mfma_f64_16x16x4 issues
// every 115-128 cycles (probe; 64 at the nominal rate), so a 16 x 32 tile is ~10k cycles,
// 4.3 us, and a second wave on the SIMD adds nothing.  v_mfma_f64_4x4x4 issues every 16.6 (1.7
// times the rate), but with its keys broadcast over the four blocks it reads and widens every
// K element four times (427 us for the four prompts of 1000), and with the dims over the blocks
// and a reduce-scatter of the shares its 32 accumulators spill 18 registers (363 us,
// bit-identical).
// Both 16x16x4 MFMAs take A[l % 16][l / 16] and B[l / 16][l % 16] from lane l and give it column
// l % 16 of the 16x16 result; register i holds row 4 (l / 16) + i for fp32 and row
// 4 i + l / 16 for fp64 (pinned on the device by an in-bounds probe):
//   S^T = K Q^T (fp64): rows are keys, columns the wave's 16 queries; k step (c, i) of
//     the contraction pairs lane slot l / 16 with dim 16 c + 4 (l / 16) + i on both
//     sides (the pairing only has to agree between A and B); register i of a lane is key
//     4 i + l / 16 of the 16-key tile;
//   O^T = V^T P^T (fp32): rows are dims, columns queries; k step j pairs slot l / 16
//     with key 4 j + l / 16, which is exactly the S^T register j a lane already holds, so
//     P needs no exchange between lanes.  Row i of tile t < 4 (D / 64) is dim
//     64 (t / 4) + 4 i + t % 4, so one 16-byte read of a V row feeds four tiles and a lane's
//     outputs are four dims in a row; the tiles past them hold 16 dims each in order.
// A query's 16 scores of a key tile sit in lanes l, l ^ 16, l ^ 32, l ^ 48.
#include <type_traits>

#include "common.h"
#include "prefill_f32.h"
#include "work_map.h"

namespace {

constexpr int kF32Waves = 4;
constexpr int kF32Threads = kF32Waves * kWave;
static_assert(kF32BlockM == 16 * kF32Waves, "16 rows a wave");
static_assert(kF32SplitMaxRows == NIA_PREFILL_F32_SPLIT_MAX_ROWS, "the header's bound");

typedef double f64x4_t __attribute__((ext_vector_type(4)));

NIA_DEVICE int f32_tok(const PrefillF32Params& p, int r) {
  return p.group == 1 ? r : key_block(r, p.group_magic, p.group_shift);
}

// Waves a SIMD (workgroups a CU) that the registers and LDS of one stage (two: PIPE) leave room for.
template <int D, bool PIPE>
constexpr int kF32PerSimd = D == 64 ? (PIPE ? 3 : 4) : D < 128 && !PIPE ? 3 : 2;

// Element kinds: fp32 rows, bf16 rows, or a paged fp8 cache (e4m3 codes with one fp32
// scale per cache row; q and o in bf16).  Every element is widened to fp32 in LDS (fp8 as
// code * row scale in fp32, the rows the fp8 format stands for), so one kernel serves the
// cache layouts the bf16 and fp8 kernels do not take: any block size, any group.
template <int D, bool PAGED, int E, bool PIPE>
__global__ __launch_bounds__(kF32Threads, (kF32PerSimd<D, PIPE>)) void prefill_f32_kernel(
    PrefillF32Params p) {
  static_assert(D % 16 == 0 && D <= 128, "head_dim a multiple of 16, at most 128");
  static_assert(E == kElemF32 || PAGED, "bf16 and fp8 elements come from a paged cache");
  constexpr int kRow = D;          // LDS row stride in floats
  constexpr int kC4 = D / 4;       // 16-byte chunks per row
  constexpr int kTiles = D / 16;   // output tiles
  constexpr int kQuads = D / 64;   // groups of four tiles read by 16-byte chunks
  constexpr int kChunks = kF32BlockN * kC4;  // per operand
  constexpr int kItems = (kChunks + kF32Threads - 1) / kF32Threads;  // of a thread
  constexpr int kAhead = D == 128;  // operands read from LDS a step ahead
  constexpr int kStages = PIPE ? 2 : 1;  // of LDS
  __shared__ __attribute__((aligned(16))) float sk[kStages][kF32BlockN * kRow];
  __shared__ __attribute__((aligned(16))) float sv[kStages][kF32BlockN * kRow];
  __shared__ int sok[kStages][kF32BlockN];  // key of the tile lies in a valid block

  int seq, hk, m0;
  f32_map(p, blockIdx.x, blockIdx.y, blockIdx.z, seq, hk, m0);
  const int G = p.group;
  const int qlen = p.decode ? 1 : p.q_len[seq];
  const int64_t qstart = p.decode ? seq : p.q_start[seq];
  const int rows = qlen * G;
  if (qlen <= 0 || m0 >= rows) return;  // uniform over the workgroup
  int klen;
  int64_t kstart = 0;
  if constexpr (PAGED) {
    int64_t c = p.ctx_len[seq];
    const int64_t cap = (int64_t)p.max_blocks * p.block_size;
    c = c < 0 ? 0 : (c > cap ? cap : c);
    klen = (int)c;
  } else {
    klen = p.k_len[seq] > 0 ? p.k_len[seq] : 0;
    kstart = p.k_start[seq];
  }
  auto tok_of = [&](int r) __attribute__((always_inline)) -> int { return f32_tok(p, r); };
  const bool causal = p.causal != NIA_CAUSAL_NONE;
  const int q_pos0 = p.causal == NIA_CAUSAL_BOTTOM_RIGHT ? klen - qlen : 0;
  int n_end = klen;
  if (causal) n_end = min(klen, max(0, q_pos0 + tok_of(min(m0 + kF32BlockM, rows) - 1) + 1));
  // keys [n_begin, n_stop) are this workgroup's
  const int tiles = (n_end + kF32BlockN - 1) / kF32BlockN;
  const int ranges = f32_ranges(tiles, p.splits);
  const int range = p.splits > 1 ? (int)blockIdx.y : 0;  // uncut: y may be a KV head
  if (range >= ranges) return;
  const int n_begin = range_tile(tiles, range, ranges) * kF32BlockN;
  const int n_stop = min(n_end, range_tile(tiles, range + 1, ranges) * kF32BlockN);

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = uniform(tid / kWave);
  const int col = lane & 15;   // the lane's query within the wave's 16
  const int slot = lane >> 4;  // k slot of the MFMA operands
  const int r = m0 + 16 * wave + col;
  const bool row_ok = r < rows;
  const int rc = row_ok ? r : 0;
  const int tok = tok_of(rc);
  const int h = hk * G + rc - tok * G;
  // keys [0, kb) are visible to this lane's query
  const int kb = row_ok ? (causal ? min(klen, max(0, q_pos0 + tok + 1)) : klen) : 0;

  // B operand of S^T: q[r][16 c + 4 slot + i] widened to fp64
  double qd[D / 4];
  {
    const int64_t qrow = (qstart + tok) * p.q_tok + (int64_t)h * p.q_head;
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      float4 u = make_float4(0.f, 0.f, 0.f, 0.f);
      if (row_ok) {
        if constexpr (E == kElemF32) {
          u = *reinterpret_cast<const float4*>(static_cast<const float*>(p.q) + qrow + 16 * c +
                                               4 * slot);
        } else {
          const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const bf16_t*>(p.q) + qrow +
                                                          16 * c + 4 * slot);
          u = make_float4(bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y));
        }
      }
      qd[4 * c + 0] = u.x;
      qd[4 * c + 1] = u.y;
      qd[4 * c + 2] = u.z;
      qd[4 * c + 3] = u.w;
    }
  }

  f32x4_t oacc[kTiles];
#pragma unroll
  for (int t = 0; t < kTiles; ++t) oacc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  double m_run = -INFINITY;  // the query's running max, log2 units
  float l_run = 0.f;         // this lane's share of the query's sum

  // Row r's 16-byte chunk c lies at c ^ swz(r): the same chunk of 16 rows, and 16 adjacent chunks
  // of one row, then fall on all 64 banks, and the chunk stays inside its row of D / 4 chunks
  // (16 or 32, 24 in groups of 8, 20 in groups of 4).
  auto swz = [](int r) __attribute__((always_inline)) -> int {
    return D % 64 == 0 ? r & 15 : (D % 32 == 0 ? (r >> 1) & 7 : (r >> 2) & 3);
  };
  const int32_t* bt = PAGED ? p.block_tables + (int64_t)seq * p.bt_stride : nullptr;
  const float* bias_row = p.bias ? p.bias + (int64_t)seq * p.bias_seq + (int64_t)h * p.bias_head +
                                       (int64_t)tok * p.bias_q
                                 : nullptr;

  // ---- staging: keys n0 .. n0 + 31 into registers (zeros past the context and in invalid
  // blocks), then into an LDS stage ------------------------------------------------------------
  // fp32 chunks; bf16 and fp8 as loaded, widened when they are written
  using Raw = std::conditional_t<E == kElemF32, float4,
                                 std::conditional_t<E == kElemBf16, uint2, uint32_t>>;
  Raw kr[kItems], vr[kItems];
  float ksr[kItems], vsr[kItems];  // fp8 row scales
  uint32_t okr = 0;                // bit i: item i's key lies in a valid block
  auto load_tile = [&](int n0) __attribute__((always_inline)) {
    okr = 0;
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const int idx = tid + i * kF32Threads;
      const int key = idx / kC4;
      const int c4 = idx - key * kC4;
      const int t = n0 + key;
      kr[i] = vr[i] = Raw{};
      ksr[i] = vsr[i] = 0.f;
      bool ok = t < klen && idx < kChunks;
      if (!ok) continue;
      int64_t ko, vo;  // element offsets of the chunks
      int64_t row = 0;
      if constexpr (PAGED) {
        const int blk = bt[t / p.block_size];
        ok = blk >= 0 && (int64_t)blk < p.num_blocks;
        row = ((int64_t)(ok ? blk : 0) * p.num_kv_heads + hk) * p.block_size + t % p.block_size;
        ko = vo = row * D + 4 * c4;
      } else {
        ko = (kstart + t) * p.k_tok + (int64_t)hk * p.k_head + 4 * c4;
        vo = (kstart + t) * p.v_tok + (int64_t)hk * p.v_head + 4 * c4;
      }
      if (!ok) continue;
      okr |= 1u << i;
      using El = std::conditional_t<E == kElemF32, float,
                                    std::conditional_t<E == kElemBf16, bf16_t, uint8_t>>;
      kr[i] = *reinterpret_cast<const Raw*>(static_cast<const El*>(p.k) + ko);
      vr[i] = *reinterpret_cast<const Raw*>(static_cast<const El*>(p.v) + vo);
      if constexpr (E == kElemFp8) {
        ksr[i] = p.k_scale[row];
        vsr[i] = p.v_scale[row];
      }
    }
  };
  auto widen = [](const Raw& w, float scale) __attribute__((always_inline)) -> float4 {
    if constexpr (E == kElemF32) {
      return w;
    } else if constexpr (E == kElemBf16) {
      return make_float4(bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y));
    } else {
      const uint32_t a = bf16x2_from_fp8x2<false>(w), b = bf16x2_from_fp8x2<true>(w);
      return make_float4(bf16_lo(a) * scale, bf16_hi(a) * scale, bf16_lo(b) * scale,
                         bf16_hi(b) * scale);
    }
  };
  auto store_tile = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const int idx = tid + i * kF32Threads;
      const int key = idx / kC4;
      const int c4 = idx - key * kC4;
      const int at = key * kRow + 4 * (c4 ^ swz(key));
      if (kChunks % kF32Threads != 0 && idx >= kChunks) break;
      *reinterpret_cast<float4*>(sk[stage] + at) = widen(kr[i], ksr[i]);
      *reinterpret_cast<float4*>(sv[stage] + at) = widen(vr[i], vsr[i]);
      if (c4 == 0) sok[stage][key] = (okr >> i) & 1u;
    }
  };

  auto compute = [&](int n0, int stage) __attribute__((always_inline)) {
    // ---- S^T = K Q^T in fp64, two 16-key tiles ----------------------------------------------
    f64x4_t s[2];
    s[0] = s[1] = f64x4_t{0.0, 0.0, 0.0, 0.0};
    const float* ks = sk[stage] + col * kRow;
    // the operands of step c + 1 are read while the products of step c run, and the two
    // tiles' chains alternate
    auto k_read = [&](int c, float4 (&a)[2]) __attribute__((always_inline)) {
      const int at = 4 * ((4 * c + slot) ^ swz(col));
      a[0] = *reinterpret_cast<const float4*>(ks + at);
      a[1] = *reinterpret_cast<const float4*>(ks + 16 * kRow + at);
    };
    float4 ka[kAhead + 1][2];
    if constexpr (kAhead) k_read(0, ka[0]);
#pragma unroll
    for (int c = 0; c < D / 16; ++c) {
      if (!kAhead || c + 1 < D / 16) k_read(c + kAhead, ka[(c + kAhead) & kAhead]);
      if constexpr (kAhead) __builtin_amdgcn_sched_barrier(0);
      const float4(&a)[2] = ka[c & kAhead];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        s[kt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[kt].x, qd[4 * c + 0], s[kt], 0, 0, 0);
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        s[kt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[kt].y, qd[4 * c + 1], s[kt], 0, 0, 0);
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        s[kt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[kt].z, qd[4 * c + 2], s[kt], 0, 0, 0);
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        s[kt] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[kt].w, qd[4 * c + 3], s[kt], 0, 0, 0);
    }
    // ---- online softmax: lane register i of tile kt is key n0 + 16 kt + 4 i + slot ----------
    double xs[2][4];
    double mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = 16 * kt + 4 * i + slot;
        const bool vis = n0 + key < kb && sok[stage][key];
        xs[kt][i] = vis ? s[kt][i] * p.scale_log2 : -INFINITY;
        if (!PAGED && p.bias && vis)
          xs[kt][i] += (double)bias_row[n0 + key] * 1.4426950408889634;
        mx = fmax(mx, xs[kt][i]);
      }
    mx = fmax(mx, __shfl_xor(mx, 16, kWave));
    mx = fmax(mx, __shfl_xor(mx, 32, kWave));
    const double mn = fmax(m_run, mx);
    if (mn > m_run) {  // lane-uniform within the query's four lanes
      const float corr = (m_run == -INFINITY) ? 0.f : fast_exp2((float)(m_run - mn));
      m_run = mn;
      l_run *= corr;
#pragma unroll
      for (int t = 0; t < kTiles; ++t) oacc[t] *= corr;
    }
    float pr[2][4];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pr[kt][i] = xs[kt][i] == -INFINITY ? 0.f : fast_exp2((float)(xs[kt][i] - m_run));
        l_run += pr[kt][i];
      }
    // ---- O^T += V^T P^T, the next key group's V read a step ahead ---------------------------
    struct VRow {
      float4 q[kQuads];
      float t[kTiles - 4 * kQuads + 1];
    };
    auto v_read = [&](int u, VRow& a) __attribute__((always_inline)) {  // keys 4 u + slot
      const float* vrow = sv[stage] + (4 * u + slot) * kRow;
      const int sw = swz(4 * u + slot);
#pragma unroll
      for (int g = 0; g < kQuads; ++g)
        a.q[g] = *reinterpret_cast<const float4*>(vrow + 4 * ((16 * g + col) ^ sw));
#pragma unroll
      for (int t = 4 * kQuads; t < kTiles; ++t) {
        const int d = 16 * t + col;
        a.t[t - 4 * kQuads] = vrow[4 * ((d >> 2) ^ sw) + (d & 3)];
      }
    };
    VRow va[kAhead + 1];
    if constexpr (kAhead) v_read(0, va[0]);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (!kAhead || u < 7) v_read(u + kAhead, va[(u + kAhead) & kAhead]);
      if constexpr (kAhead) __builtin_amdgcn_sched_barrier(0);
      const VRow& a = va[u & kAhead];
      const float pu = pr[u >> 2][u & 3];
#pragma unroll
      for (int g = 0; g < kQuads; ++g) {
        oacc[4 * g + 0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.q[g].x, pu, oacc[4 * g + 0], 0, 0, 0);
        oacc[4 * g + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.q[g].y, pu, oacc[4 * g + 1], 0, 0, 0);
        oacc[4 * g + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.q[g].z, pu, oacc[4 * g + 2], 0, 0, 0);
        oacc[4 * g + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.q[g].w, pu, oacc[4 * g + 3], 0, 0, 0);
      }
#pragma unroll
      for (int t = 4 * kQuads; t < kTiles; ++t)
        oacc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.t[t - 4 * kQuads], pu, oacc[t], 0, 0, 0);
    }
  };

  if constexpr (kStages == 1) {
    for (int n0 = n_begin; n0 < n_stop; n0 += kF32BlockN) {
      __syncthreads();
      load_tile(n0);
      store_tile(0);
      __syncthreads();
      if (wave_any(n0 < kb)) compute(n0, 0);
    }
  } else if (n_begin < n_stop) {
    load_tile(n_begin);
    store_tile(0);
    __syncthreads();
    int stage = 0;
    for (int n0 = n_begin; n0 < n_stop; n0 += kF32BlockN) {
      const bool more = n0 + kF32BlockN < n_stop;
      if (more) load_tile(n0 + kF32BlockN);
      if (wave_any(n0 < kb)) compute(n0, stage);  // else no query of this wave sees the tile
      if (more) store_tile(stage ^ 1);
      __syncthreads();
      stage ^= 1;
    }
  }

  // ---- normalise and store: lane l holds rows 4 slot + i of every tile for query col --------
  l_run += __shfl_xor(l_run, 16, kWave);
  l_run += __shfl_xor(l_run, 32, kWave);
  if (!row_ok) return;
  if (ranges > 1) {  // un-normalised, for prefill_f32_merge_kernel
    const int64_t prow =
        ((int64_t)range * gridDim.x + blockIdx.x) * kF32BlockM + (r - m0);
    if (slot == 0) {
      p.part_m[prow] = m_run;
      p.part_l[prow] = l_run;
    }
    float* po = p.part_o + prow * D;
#pragma unroll
    for (int g = 0; g < kQuads; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4*>(po + 64 * g + 4 * (4 * slot + i)) =
            make_float4(oacc[4 * g][i], oacc[4 * g + 1][i], oacc[4 * g + 2][i], oacc[4 * g + 3][i]);
#pragma unroll
    for (int t = 4 * kQuads; t < kTiles; ++t)
      *reinterpret_cast<float4*>(po + 16 * t + 4 * slot) =
          make_float4(oacc[t][0], oacc[t][1], oacc[t][2], oacc[t][3]);
    return;
  }
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  const int64_t orow = (qstart + tok) * p.o_tok + (int64_t)h * p.o_head;
  auto store4 = [&](int d, float a, float b, float c, float e) __attribute__((always_inline)) {
    if constexpr (E == kElemF32)
      *reinterpret_cast<float4*>(static_cast<float*>(p.o) + orow + d) =
          make_float4(a * inv, b * inv, c * inv, e * inv);
    else
      *reinterpret_cast<uint2*>(static_cast<bf16_t*>(p.o) + orow + d) =
          make_uint2(pack_bf16x2(a * inv, b * inv), pack_bf16x2(c * inv, e * inv));
  };
#pragma unroll
  for (int g = 0; g < kQuads; ++g)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      store4(64 * g + 4 * (4 * slot + i), oacc[4 * g][i], oacc[4 * g + 1][i], oacc[4 * g + 2][i],
             oacc[4 * g + 3][i]);
#pragma unroll
  for (int t = 4 * kQuads; t < kTiles; ++t)
    store4(16 * t + 4 * slot, oacc[t][0], oacc[t][1], oacc[t][2], oacc[t][3]);
}

// Merges the ranges' partials of the fp32 output rows that have more than one: 32 lanes a row,
// four dims each.
template <int D, bool PAGED>
__global__ __launch_bounds__(kF32Threads) void prefill_f32_merge_kernel(PrefillF32Params p) {
  constexpr int kLanes = 32;
  int seq, hk, m0;
  f32_map(p, blockIdx.x, blockIdx.y, blockIdx.z, seq, hk, m0);
  const int qlen = p.q_len[seq];
  const int rows = qlen * p.group;
  const int rr = blockIdx.y * (kF32Threads / kLanes) + threadIdx.x / kLanes;  // of the block
  if (qlen <= 0 || m0 + rr >= rows) return;
  int klen;
  if constexpr (PAGED) {
    int64_t c = p.ctx_len[seq];
    const int64_t cap = (int64_t)p.max_blocks * p.block_size;
    klen = (int)(c < 0 ? 0 : (c > cap ? cap : c));
  } else {
    klen = p.k_len[seq] > 0 ? p.k_len[seq] : 0;
  }
  const int q_pos0 = p.causal == NIA_CAUSAL_BOTTOM_RIGHT ? klen - qlen : 0;
  int n_end = klen;
  if (p.causal != NIA_CAUSAL_NONE)
    n_end = min(klen, max(0, q_pos0 + f32_tok(p, min(m0 + kF32BlockM, rows) - 1) + 1));
  const int ranges = f32_ranges((n_end + kF32BlockN - 1) / kF32BlockN, p.splits);
  const int d = 4 * (threadIdx.x % kLanes);
  if (ranges == 1 || d >= D) return;
  const int64_t prow = (int64_t)blockIdx.x * kF32BlockM + rr;
  const int64_t step = (int64_t)gridDim.x * kF32BlockM;
  double m = -INFINITY;
  float l = 0.f;
  f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < ranges; ++s) m = fmax(m, p.part_m[s * step + prow]);
  for (int s = 0; s < ranges; ++s) {
    const int64_t pr = s * step + prow;
    const double ms = p.part_m[pr];
    const f32x4_t o = *reinterpret_cast<const f32x4_t*>(p.part_o + pr * D + d);
    // no visible key: m = -inf, l = 0; NaN scores leave m and make l NaN, and a NaN in o stays
    // one at any weight, as in an uncut call
    const bool any = ms != -INFINITY;
    const float w = any ? fast_exp2((float)(ms - m)) : 0.f;
    l = fmaf(p.part_l[pr], w, l);
    if (any) acc += o * w;
  }
  const float inv = l != 0.f ? 1.f / l : 0.f;
  const int tok = f32_tok(p, m0 + rr);
  float* o = static_cast<float*>(p.o) + (p.q_start[seq] + (int64_t)tok) * p.o_tok +
             (int64_t)(hk * p.group + m0 + rr - tok * p.group) * p.o_head + d;
  *reinterpret_cast<float4*>(o) = make_float4(acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv);
}

template <int D, bool PAGED, int E>
void launch_f32(const PrefillF32Params& p, dim3 grid, hipStream_t s) {
  if constexpr (PAGED && D < 128) {
    const int64_t nwg = (int64_t)grid.x * grid.y * grid.z;
    if (p.decode && f32_two_stages(D, nwg, (int64_t)p.max_blocks * p.block_size)) {
      nia_launch((prefill_f32_kernel<D, PAGED, E, true>), grid, dim3(kF32Threads), s, p);
      return;
    }
  }
  nia_launch((prefill_f32_kernel<D, PAGED, E, D == 128>), grid, dim3(kF32Threads), s, p);
}

template <int D, bool PAGED>
void launch_f32_split(const PrefillF32Params& p, dim3 grid, hipStream_t s) {
  launch_f32<D, PAGED, kElemF32>(p, dim3(grid.x, (unsigned)p.splits), s);
  nia_launch((prefill_f32_merge_kernel<D, PAGED>), dim3(grid.x, kF32BlockM * 32 / kF32Threads),
             dim3(kF32Threads), s, p);
}

}  // namespace

size_t prefill_f32_split_bytes(int32_t num_seqs, int64_t max_q_len, int64_t max_k_len,
                               int32_t num_heads, int32_t num_kv_heads, int head_dim) {
  int32_t blocks;
  int64_t rows = max_q_len * (num_heads / num_kv_heads);
  if (rows > INT32_MAX) rows = INT32_MAX;
  const int64_t nwg = f32_grid((int64_t)num_seqs * num_kv_heads, rows, blocks);
  const int64_t sure = num_seqs == 1 ? max_q_len * num_heads : 0;
  return f32_split_bytes(nwg, f32_split_count(nwg, max_k_len, sure), head_dim);
}

int32_t launch_prefill_f32(PrefillF32Params& p, bool paged, int head_dim, int num_seqs,
                           int max_q_len, hipStream_t stream, int elem, void* ws,
                           size_t ws_bytes, int64_t max_k_len) {
  if (num_seqs > 65535 || p.num_heads > 65535) return NIA_ERR_UNSUPPORTED;
  if (elem != kElemF32 && (!paged || elem != kElemBf16) && (!paged || elem != kElemFp8))
    return NIA_ERR_UNSUPPORTED;
  if (elem == kElemFp8 && (head_dim != 128 || !p.k_scale || !p.v_scale))
    return NIA_ERR_UNSUPPORTED;
  // row numbers are ints
  int64_t rows = (int64_t)(p.decode ? 1 : max_q_len) * p.group;
  if (rows > INT32_MAX) rows = INT32_MAX;
  block_divisor(p.group, p.group_magic, p.group_shift);
  const int64_t groups = (int64_t)num_seqs * p.num_kv_heads;
  const int64_t nwg = f32_grid(groups, rows, p.num_m_blocks);
  p.groups = (int32_t)at_most(groups, kMaxGroups);  // 1-D: no more than its workgroups
  p.splits = 1;
  if (ws && elem == kElemF32 && !p.decode) {
    const int64_t sure = num_seqs == 1 ? (int64_t)max_q_len * p.num_heads : 0;
    const int32_t n = f32_split_count(nwg, max_k_len, sure);
    if (n > 1 && f32_split_bytes(nwg, n, head_dim) <= ws_bytes) {
      const size_t parts = (size_t)nwg * n * kF32BlockM;
      p.splits = n;
      p.part_m = (double*)ws;
      p.part_o = (float*)(p.part_m + parts);
      p.part_l = p.part_o + parts * head_dim;
    }
  }
  p.level_run = f32_run(nwg, p.num_m_blocks, p.causal == NIA_CAUSAL_TOP_LEFT, p.splits > 1);
  const dim3 grid = p.level_run ? dim3((unsigned)nwg)
                                : dim3((unsigned)p.num_m_blocks, (unsigned)p.num_kv_heads,
                                       (unsigned)num_seqs);
  if (elem == kElemFp8) {
    launch_f32<128, true, kElemFp8>(p, grid, stream);
    return hipGetLastError() == hipSuccess ? NIA_OK : NIA_ERR_LAUNCH;
  }
  switch (head_dim) {
#define NIA_F32_CASE(DD)                                                                      \
  case DD:                                                                                    \
    if (p.splits > 1 && paged)                                                                \
      launch_f32_split<DD, true>(p, grid, stream);                                            \
    else if (p.splits > 1)                                                                    \
      launch_f32_split<DD, false>(p, grid, stream);                                           \
    else if (!paged)                                                                          \
      launch_f32<DD, false, kElemF32>(p, grid, stream);                                       \
    else if (elem == kElemF32)                                                                \
      launch_f32<DD, true, kElemF32>(p, grid, stream);                                        \
    else                                                                                      \
      launch_f32<DD, true, kElemBf16>(p, grid, stream);                                       \
    break;
    NIA_F32_CASE(64)
    NIA_F32_CASE(80)
    NIA_F32_CASE(96)
    NIA_F32_CASE(128)
#undef NIA_F32_CASE
    default:
      return NIA_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? NIA_OK : NIA_ERR_LAUNCH;
}
