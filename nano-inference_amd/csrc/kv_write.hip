// KV-cache write (scatter new K/V rows into physical slots), gfx950.
//
// Replaces the per-token Python loop of the reference,
// src/nano_inference/layers/attention.py:267-278, which does one host sync and
// two indexed copies per token.  Here one launch moves every token: each lane
// copies 16 bytes of K and 16 bytes of V, so a (token, kv-head) row of 128 bf16
// is 16 lanes and a wave covers 4 rows.  The copy is a bit copy (uint4), so the
// result is bit-exact whatever the element type.
//
// HBM traffic per token: read 2 * H_kv * D * s, write 2 * H_kv * D * s, plus the
// 8-byte slot; the kernel is latency-bound at decode sizes (tens of tokens) and
// bandwidth-bound at prefill sizes.
#include <type_traits>

#include "common.h"
#include "prefill_args.h"
#include "work_map.h"

namespace {

// VEC_BYTES: bytes per lane per copy (16 when every row start is 16-byte
// aligned, else the element size).
template <int VEC_BYTES>
__global__ __launch_bounds__(256) void kv_write_kernel(
    const uint8_t* __restrict__ k, int64_t k_tok_stride_b, int64_t k_head_stride_b,
    const uint8_t* __restrict__ v, int64_t v_tok_stride_b, int64_t v_head_stride_b,
    uint8_t* __restrict__ k_cache, uint8_t* __restrict__ v_cache,
    const int64_t* __restrict__ slot_mapping, int32_t num_tokens, int32_t num_kv_heads,
    int32_t row_bytes, int32_t block_size, int64_t num_slots) {
  using vec_t = typename std::conditional<
      VEC_BYTES == 16, uint4,
      typename std::conditional<VEC_BYTES == 8, uint2,
                                typename std::conditional<VEC_BYTES == 4, uint32_t,
                                                          uint16_t>::type>::type>::type;
  // 32-bit indexing: the host guarantees num_tokens * num_kv_heads * row_bytes < 2^31.
  const int vec_per_row = row_bytes / VEC_BYTES;
  const int vec_per_tok = vec_per_row * num_kv_heads;
  const int total = vec_per_tok * num_tokens;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
    const int tok = i / vec_per_tok;
    const int rem = i - tok * vec_per_tok;
    const int head = rem / vec_per_row;
    const int c = rem - head * vec_per_row;
    const int64_t slot = slot_mapping[tok];
    if (slot < 0 || slot >= num_slots) continue;
    const int64_t blk = slot / block_size;
    const int64_t off = slot - blk * block_size;
    const int64_t dst = (((blk * num_kv_heads + head) * block_size + off) * row_bytes) +
                        (int64_t)c * VEC_BYTES;
    const vec_t kv = *reinterpret_cast<const vec_t*>(k + (int64_t)tok * k_tok_stride_b +
                                                     head * k_head_stride_b + c * VEC_BYTES);
    const vec_t vv = *reinterpret_cast<const vec_t*>(v + (int64_t)tok * v_tok_stride_b +
                                                     head * v_head_stride_b + c * VEC_BYTES);
    *reinterpret_cast<vec_t*>(k_cache + dst) = kv;
    *reinterpret_cast<vec_t*>(v_cache + dst) = vv;
  }
}

bool aligned(const void* p, int64_t a) { return ((uintptr_t)p % (uintptr_t)a) == 0; }

}  // namespace

extern "C" int32_t nia_kv_write(const void* k, int64_t k_tok_stride, int64_t k_head_stride,
                                const void* v, int64_t v_tok_stride, int64_t v_head_stride,
                                void* k_cache, void* v_cache, const int64_t* slot_mapping,
                                int32_t num_tokens, int32_t num_kv_heads, int32_t head_dim,
                                int32_t block_size, int64_t num_blocks, int32_t dtype,
                                void* stream) {
  if (num_tokens < 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size <= 0 ||
      num_blocks < 0)
    return NIA_ERR_INVALID_ARGUMENT;
  if (dtype != NIA_DTYPE_BF16 && dtype != NIA_DTYPE_F32) return NIA_ERR_UNSUPPORTED;
  if (num_tokens == 0 || num_blocks == 0) return NIA_OK;
  if (!k || !v || !k_cache || !v_cache || !slot_mapping) return NIA_ERR_INVALID_ARGUMENT;
  const int64_t es = dtype == NIA_DTYPE_BF16 ? 2 : 4;
  const int64_t row_bytes = head_dim * es;
  const int64_t kt = k_tok_stride * es, kh = k_head_stride * es;
  const int64_t vt = v_tok_stride * es, vh = v_head_stride * es;
  auto fits = [&](int64_t a) {
    return row_bytes % a == 0 && kt % a == 0 && kh % a == 0 && vt % a == 0 && vh % a == 0 &&
           aligned(k, a) && aligned(v, a) && aligned(k_cache, a) && aligned(v_cache, a);
  };
  const int64_t num_slots = num_blocks * block_size;
  const int64_t rows = (int64_t)num_tokens * num_kv_heads;
  if (rows * row_bytes >= ((int64_t)1 << 31)) return NIA_ERR_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  auto launch = [&](auto kernel, int vec) {
    const int64_t work = rows * (row_bytes / vec);
    const int64_t blocks = (work + 255) / 256;
    const unsigned grid = (unsigned)(blocks < 65536 ? blocks : 65536);
    nia_launch(kernel, dim3(grid), dim3(256), s, (const uint8_t*)k, kt, kh,
               (const uint8_t*)v, vt, vh, (uint8_t*)k_cache, (uint8_t*)v_cache,
               slot_mapping, num_tokens, num_kv_heads, (int32_t)row_bytes, block_size,
               num_slots);
  };
  if (fits(16))
    launch(kv_write_kernel<16>, 16);
  else if (fits(8))
    launch(kv_write_kernel<8>, 8);
  else if (fits(4))
    launch(kv_write_kernel<4>, 4);
  else if (fits(2))
    launch(kv_write_kernel<2>, 2);
  else
    return NIA_ERR_MISALIGNED;
  return hipGetLastError() == hipSuccess ? NIA_OK : NIA_ERR_LAUNCH;
}

// ---------------------------------------------------------------------------------
// fp8 KV-cache write: each (token, KV head) row of 128 values is stored as OCP e4m3
// codes with one fp32 scale, scale = max |x| / 448, code = e4m3(x / scale) (round to
// nearest even; the row maximum lands on 448 exactly, a zero row stores scale 0).
// One wave per row (K rows, then V rows): lane l quantises dims 2l and 2l + 1, the
// row maximum is a wave reduction, and the 128 codes leave as one coalesced store.
// ---------------------------------------------------------------------------------
namespace {

constexpr int kFp8Rows = 4;  // rows (waves) per workgroup

template <typename T>
__global__ __launch_bounds__(kFp8Rows * kWave) void kv_write_fp8_kernel(
    const T* __restrict__ k, int64_t k_tok, int64_t k_head, const T* __restrict__ v,
    int64_t v_tok, int64_t v_head, uint8_t* __restrict__ k_cache, uint8_t* __restrict__ v_cache,
    float* __restrict__ k_scale, float* __restrict__ v_scale,
    const int64_t* __restrict__ slot_mapping, int32_t num_tokens, int32_t num_kv_heads,
    int32_t block_size, int64_t num_slots) {
  constexpr int D = 128;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = (int64_t)blockIdx.x * kFp8Rows + (threadIdx.x >> 6);
  const int64_t rows = (int64_t)num_tokens * num_kv_heads;
  if (row >= 2 * rows) return;
  const bool is_v = row >= rows;
  const int64_t r = is_v ? row - rows : row;
  const int tok = (int)(r / num_kv_heads);
  const int head = (int)(r - (int64_t)tok * num_kv_heads);
  const int64_t slot = slot_mapping[tok];
  if (slot < 0 || slot >= num_slots) return;
  const T* src = is_v ? v + tok * v_tok + head * v_head : k + tok * k_tok + head * k_head;
  const float x0 = (float)src[2 * lane];
  const float x1 = (float)src[2 * lane + 1];
  float amax = fmaxf(fabsf(x0), fabsf(x1));
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) amax = fmaxf(amax, __shfl_xor(amax, off, kWave));
  const float scale = amax / kE4m3Max;
  const uint32_t codes = scale > 0.f ? fp8x2_from_f32(x0 / scale, x1 / scale) : 0u;
  const int64_t blk = slot / block_size;
  const int64_t off = slot - blk * block_size;
  const int64_t dst_row = (blk * num_kv_heads + head) * block_size + off;
  uint8_t* dst = (is_v ? v_cache : k_cache) + dst_row * D;
  reinterpret_cast<uint16_t*>(dst)[lane] = (uint16_t)codes;
  if (lane == 0) (is_v ? v_scale : k_scale)[dst_row] = scale;
}

}  // namespace

extern "C" int32_t nia_kv_write_fp8(const void* k, int64_t k_tok_stride, int64_t k_head_stride,
                                    const void* v, int64_t v_tok_stride, int64_t v_head_stride,
                                    void* k_cache, void* v_cache, float* k_scale, float* v_scale,
                                    const int64_t* slot_mapping, int32_t num_tokens,
                                    int32_t num_kv_heads, int32_t head_dim, int32_t block_size,
                                    int64_t num_blocks, int32_t dtype, void* stream) {
  if (num_tokens < 0 || num_kv_heads <= 0 || head_dim <= 0 || block_size <= 0 ||
      num_blocks < 0)
    return NIA_ERR_INVALID_ARGUMENT;
  if (head_dim != 128 || (dtype != NIA_DTYPE_BF16 && dtype != NIA_DTYPE_F32))
    return NIA_ERR_UNSUPPORTED;
  if (num_tokens == 0 || num_blocks == 0) return NIA_OK;
  if (!k || !v || !k_cache || !v_cache || !k_scale || !v_scale || !slot_mapping)
    return NIA_ERR_INVALID_ARGUMENT;
  if (!aligned(k_cache, 2) || !aligned(v_cache, 2)) return NIA_ERR_MISALIGNED;
  const int64_t rows = 2 * (int64_t)num_tokens * num_kv_heads;
  const int64_t groups = (rows + kFp8Rows - 1) / kFp8Rows;
  if (groups > kMaxGroups) return NIA_ERR_UNSUPPORTED;
  const int64_t num_slots = num_blocks * block_size;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == NIA_DTYPE_BF16)
    nia_launch(kv_write_fp8_kernel<bf16_t>, dim3((unsigned)groups), dim3(kFp8Rows * kWave), s,
               (const bf16_t*)k, k_tok_stride, k_head_stride, (const bf16_t*)v, v_tok_stride,
               v_head_stride, (uint8_t*)k_cache, (uint8_t*)v_cache, k_scale, v_scale,
               slot_mapping, num_tokens, num_kv_heads, block_size, num_slots);
  else
    nia_launch(kv_write_fp8_kernel<float>, dim3((unsigned)groups), dim3(kFp8Rows * kWave), s,
               (const float*)k, k_tok_stride, k_head_stride, (const float*)v, v_tok_stride,
               v_head_stride, (uint8_t*)k_cache, (uint8_t*)v_cache, k_scale, v_scale,
               slot_mapping, num_tokens, num_kv_heads, block_size, num_slots);
  return hipGetLastError() == hipSuccess ? NIA_OK : NIA_ERR_LAUNCH;
}

// ---------------------------------------------------------------------------------
// fp8 cache -> contiguous bf16 rows: sequence s's keys [0, context_lens[s]) gathered
// through its block table and dequantised (code * row scale, rounded to bf16) into
// out_k / out_v.  Feeds the varlen prefill kernel for chunked prefill over an fp8 cache.
//
// Bound by HBM (a byte and a share of a scale in, two bytes out per element).  A workgroup
// takes up to kGatherItems 16-code pieces of one cache block, which lie one after another
// in the cache ([KV head][row][128]), two to a thread with the K and V loads of both in
// flight together: 16-byte loads, two 16-byte stores (four to a thread: 4 us slower).  A
// row a wave with 2-byte loads before: 148 us for 33k keys of 8 heads, 1.4 TB/s; now
// 43-48 us, 4.2-4.7 TB/s.  The chunked prefill of eight 512-row chunks over those keys
// takes 383-387 us before, 282-291 now, of which 240 is the attention.
// ---------------------------------------------------------------------------------
namespace {

constexpr int kGatherThreads = 256;
constexpr int kGatherUnroll = 2;
constexpr int kGatherItems = kGatherThreads * kGatherUnroll;

struct GatherParams {
  const uint8_t* k_cache;
  const uint8_t* v_cache;
  const float* k_scale;
  const float* v_scale;
  const int32_t* block_tables;
  const int64_t* context_lens;
  bf16_t* out_k;  // row of key t, head h of sequence s: s * seq + h * head + t * tok elements on
  bf16_t* out_v;
  int64_t seq, head, tok;
  int64_t num_blocks;
  int32_t bt_stride, max_blocks, num_kv_heads, block_size;
  int32_t parts;     // workgroups per block
  int32_t* k_start;  // optional: first row (s * start) and key count of each sequence
  int32_t* k_len;
  int64_t start;
};

// VEC: 16-byte accesses; else the 2-byte loads and 4-byte stores that any accepted pointer
// allows.
template <bool VEC>
__global__ __launch_bounds__(kGatherThreads) void dequant_gather_fp8_kernel(GatherParams p) {
  constexpr int D = 128;
  const int s = blockIdx.y;
  const uint32_t id = blockIdx.z * gridDim.x + blockIdx.x;  // past the table: past the context
  const uint32_t jb = id / (uint32_t)p.parts;
  const int part = (int)(id - jb * (uint32_t)p.parts);
  int64_t ctx = p.context_lens[s];
  const int64_t cap = (int64_t)p.max_blocks * p.block_size;
  ctx = ctx < 0 ? 0 : (ctx > cap ? cap : ctx);
  if (p.k_start && id == 0 && threadIdx.x == 0) {
    p.k_start[s] = (int32_t)(s * p.start);
    p.k_len[s] = (int32_t)ctx;
  }
  const int64_t t0 = (int64_t)jb * p.block_size;
  if (t0 >= ctx) return;
  const int blk = p.block_tables[(int64_t)s * p.bt_stride + jb];
  const bool ok = blk >= 0 && blk < p.num_blocks;  // an invalid block id reads as zeros
  const uint32_t per_head = (uint32_t)p.block_size * (D / 16);  // pieces of a head's rows
  const uint32_t pieces = per_head * (uint32_t)p.num_kv_heads;
  const int64_t base = (int64_t)(ok ? blk : 0) * p.num_kv_heads * p.block_size;
  uint4 kc[kGatherUnroll], vc[kGatherUnroll];
  float ks[kGatherUnroll], vs[kGatherUnroll];
  int64_t dst[kGatherUnroll];  // negative: nothing to write
  auto load = [](const uint8_t* src) __attribute__((always_inline)) -> uint4 {
    if constexpr (VEC) {
      return *reinterpret_cast<const uint4*>(src);
    } else {
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint16_t* h = reinterpret_cast<const uint16_t*>(src) + 2 * i;
        w[i] = (uint32_t)h[0] | (uint32_t)h[1] << 16;
      }
      return make_uint4(w[0], w[1], w[2], w[3]);
    }
  };
#pragma unroll
  for (int u = 0; u < kGatherUnroll; ++u) {
    const uint32_t i = (uint32_t)part * kGatherItems + u * kGatherThreads + threadIdx.x;
    const uint32_t head = i / per_head;
    const uint32_t rem = i - head * per_head;
    const uint32_t row = rem / (D / 16), piece = rem % (D / 16);
    const int64_t t = t0 + row;
    dst[u] = -1;
    kc[u] = vc[u] = make_uint4(0u, 0u, 0u, 0u);
    ks[u] = vs[u] = 0.f;
    if (i >= pieces || t >= ctx) continue;
    dst[u] = s * p.seq + head * p.head + t * p.tok + 16 * piece;
    if (!ok) continue;
    const int64_t src = base + (int64_t)head * p.block_size + row;
    kc[u] = load(p.k_cache + src * D + 16 * piece);
    vc[u] = load(p.v_cache + src * D + 16 * piece);
    ks[u] = p.k_scale[src];
    vs[u] = p.v_scale[src];
  }
  auto widen = [](uint32_t w, float scale) __attribute__((always_inline)) -> uint2 {
    const uint32_t a = bf16x2_from_fp8x2<false>(w), b = bf16x2_from_fp8x2<true>(w);
    return make_uint2(pack_bf16x2(bf16_lo(a) * scale, bf16_hi(a) * scale),
                      pack_bf16x2(bf16_lo(b) * scale, bf16_hi(b) * scale));
  };
  auto store = [&](bf16_t* out, const uint4& c, float scale) __attribute__((always_inline)) {
    const uint2 a = widen(c.x, scale), b = widen(c.y, scale), d = widen(c.z, scale),
                e = widen(c.w, scale);
    if constexpr (VEC) {
      reinterpret_cast<uint4*>(out)[0] = make_uint4(a.x, a.y, b.x, b.y);
      reinterpret_cast<uint4*>(out)[1] = make_uint4(d.x, d.y, e.x, e.y);
    } else {
      const uint32_t w[8] = {a.x, a.y, b.x, b.y, d.x, d.y, e.x, e.y};
#pragma unroll
      for (int i = 0; i < 8; ++i) reinterpret_cast<uint32_t*>(out)[i] = w[i];
    }
  };
#pragma unroll
  for (int u = 0; u < kGatherUnroll; ++u) {
    if (dst[u] < 0) continue;
    store(p.out_k + dst[u], kc[u], ks[u]);
    store(p.out_v + dst[u], vc[u], vs[u]);
  }
}

int32_t launch_gather(GatherParams& p, int32_t batch, hipStream_t stream) {
  const int64_t pieces = (int64_t)p.num_kv_heads * p.block_size * 8;
  if (pieces >= ((int64_t)1 << 31)) return NIA_ERR_UNSUPPORTED;
  p.parts = (int32_t)((pieces + kGatherItems - 1) / kGatherItems);
  const int64_t groups = (int64_t)p.max_blocks * p.parts;
  if (groups >= ((int64_t)1 << 31)) return NIA_ERR_UNSUPPORTED;
  // a table too wide for one dimension: over two
  const int64_t z = (groups + kMaxGroups - 1) / kMaxGroups;
  const bool vec = aligned(p.k_cache, 16) && aligned(p.v_cache, 16) && aligned(p.out_k, 16) &&
                   aligned(p.out_v, 16);
  const dim3 grid((unsigned)((groups + z - 1) / z), (unsigned)batch, (unsigned)z);
  if (vec)
    nia_launch(dequant_gather_fp8_kernel<true>, grid, dim3(kGatherThreads), stream, p);
  else
    nia_launch(dequant_gather_fp8_kernel<false>, grid, dim3(kGatherThreads), stream, p);
  return hipGetLastError() == hipSuccess ? NIA_OK : NIA_ERR_LAUNCH;
}

// The checks and parameters that both entry points below share; out_k / out_v and their
// strides are the caller's.
int32_t gather_params(GatherParams& p, const void* k_cache, const void* v_cache,
                      const float* k_scale, const float* v_scale, const int32_t* block_tables,
                      int32_t bt_stride, int32_t max_blocks, const int64_t* context_lens,
                      int32_t num_kv_heads, int32_t block_size, int64_t num_blocks, void* out_k,
                      void* out_v) {
  if (!k_cache || !v_cache || !k_scale || !v_scale || !block_tables || !context_lens ||
      !out_k || !out_v)
    return NIA_ERR_INVALID_ARGUMENT;
  if (!aligned(k_cache, 2) || !aligned(v_cache, 2) || !aligned(out_k, 4) || !aligned(out_v, 4))
    return NIA_ERR_MISALIGNED;
  p.k_cache = (const uint8_t*)k_cache;
  p.v_cache = (const uint8_t*)v_cache;
  p.k_scale = k_scale;
  p.v_scale = v_scale;
  p.block_tables = block_tables;
  p.context_lens = context_lens;
  p.out_k = (bf16_t*)out_k;
  p.out_v = (bf16_t*)out_v;
  p.num_blocks = num_blocks;
  p.bt_stride = bt_stride;
  p.max_blocks = max_blocks;
  p.num_kv_heads = num_kv_heads;
  p.block_size = block_size;
  return NIA_OK;
}

}  // namespace

extern "C" int32_t nia_dequant_gather_fp8(const void* k_cache, const void* v_cache,
                                          const float* k_scale, const float* v_scale,
                                          const int32_t* block_tables, int32_t bt_stride,
                                          int32_t max_blocks_per_seq,
                                          const int64_t* context_lens, int32_t batch,
                                          int32_t num_kv_heads, int32_t head_dim,
                                          int32_t block_size, int64_t num_blocks, void* out_k,
                                          void* out_v, int64_t seq_stride, void* stream) {
  if (batch < 0 || num_kv_heads <= 0 || max_blocks_per_seq < 0 ||
      bt_stride < max_blocks_per_seq || block_size <= 0 || num_blocks < 0)
    return NIA_ERR_INVALID_ARGUMENT;
  if (head_dim != 128) return NIA_ERR_UNSUPPORTED;
  if (batch == 0 || max_blocks_per_seq == 0) return NIA_OK;
  if (seq_stride < (int64_t)max_blocks_per_seq * block_size) return NIA_ERR_INVALID_ARGUMENT;
  if (batch > 65535) return NIA_ERR_UNSUPPORTED;
  GatherParams p{};
  const int32_t st =
      gather_params(p, k_cache, v_cache, k_scale, v_scale, block_tables, bt_stride,
                    max_blocks_per_seq, context_lens, num_kv_heads, block_size, num_blocks, out_k,
                    out_v);
  if (st != NIA_OK) return st;
  p.head = head_dim;
  p.tok = (int64_t)num_kv_heads * head_dim;
  p.seq = seq_stride * p.tok;
  return launch_gather(p, batch, (hipStream_t)stream);
}

// Chunked prefill over an fp8 cache: the gather above into the workspace, then nia_prefill
// over its rows ([key][KV head][128]; head by head measured the same).  The gather also
// writes each sequence's first row and key count, which took four small launches.
namespace {

size_t fp8_index_bytes(int32_t num_seqs) { return ((size_t)num_seqs * 8 + 255) / 256 * 256; }

}  // namespace

extern "C" size_t nia_prefill_paged_fp8_workspace_size(int32_t num_seqs, int32_t max_q_len,
                                                       int32_t num_heads, int32_t num_kv_heads,
                                                       int32_t max_blocks_per_seq,
                                                       int32_t block_size, int32_t head_dim,
                                                       int32_t causal) {
  if (num_seqs <= 0 || num_kv_heads <= 0 || max_blocks_per_seq < 0 || block_size <= 0 ||
      head_dim <= 0)
    return 0;
  return fp8_index_bytes(num_seqs) + 2 * (size_t)num_seqs * max_blocks_per_seq * block_size *
                                         num_kv_heads * head_dim * sizeof(bf16_t) +
         nia_prefill_split_workspace_size(num_seqs, max_q_len,
                                          (int64_t)max_blocks_per_seq * block_size, num_heads,
                                          num_kv_heads, head_dim, causal, NIA_DTYPE_BF16);
}

extern "C" int32_t nia_prefill_paged_fp8(
    void* out, int64_t out_tok_stride, int64_t out_head_stride, const void* q,
    int64_t q_tok_stride, int64_t q_head_stride, const void* k_cache, const void* v_cache,
    const float* k_scale, const float* v_scale, const int32_t* block_tables, int32_t bt_stride,
    int32_t max_blocks_per_seq, const int32_t* q_start, const int32_t* q_len,
    const int64_t* context_lens, int32_t num_seqs, int32_t max_q_len, int32_t num_heads,
    int32_t num_kv_heads, int32_t head_dim, int32_t block_size, int64_t num_blocks, float scale,
    int32_t causal, void* workspace, size_t workspace_bytes, void* stream) {
  if (max_blocks_per_seq < 0 || bt_stride < max_blocks_per_seq || block_size <= 0 ||
      num_blocks < 0)
    return NIA_ERR_INVALID_ARGUMENT;
  if (head_dim != 128) return NIA_ERR_UNSUPPORTED;
  const int64_t rows = (int64_t)max_blocks_per_seq * block_size;  // of a sequence
  const int64_t tok = (int64_t)num_kv_heads * head_dim;
  // All that the attention refuses is refused before the gather is launched.  Its key rows and
  // their index lie in the workspace: 256 stands for an aligned address in it.
  const void* in_ws = (const void*)256;
  bool empty = false;
  int32_t st = check_prefill_args(
      out, out_tok_stride, out_head_stride, q, q_tok_stride, q_head_stride, in_ws, tok, head_dim,
      in_ws, tok, head_dim, q_start, q_len, (const int32_t*)in_ws, (const int32_t*)in_ws, num_seqs,
      max_q_len, num_heads, num_kv_heads, head_dim, scale, causal, NIA_DTYPE_BF16, nullptr, 0, 0,
      0, empty);
  if (st != NIA_OK || empty) return st;
  // a table without blocks leaves no key rows to attend
  if (max_blocks_per_seq == 0) return NIA_ERR_INVALID_ARGUMENT;
  // the sequences' first rows are int32
  if (num_seqs > 65535 || rows > INT32_MAX || rows * num_seqs > INT32_MAX)
    return NIA_ERR_UNSUPPORTED;
  uint8_t* ws = (uint8_t*)workspace;
  const size_t half = (size_t)num_seqs * rows * num_kv_heads * head_dim * sizeof(bf16_t);
  if (!ws || workspace_bytes < fp8_index_bytes(num_seqs) + 2 * half) return NIA_ERR_WORKSPACE;
  if (!aligned(ws, 256)) return NIA_ERR_MISALIGNED;
  int32_t* k_start = (int32_t*)ws;
  int32_t* k_len = k_start + num_seqs;
  uint8_t* keys = ws + fp8_index_bytes(num_seqs);
  uint8_t* vals = keys + half;
  uint8_t* split = vals + half;
  const size_t split_bytes = workspace_bytes - (size_t)(split - ws);
  GatherParams p{};
  st = gather_params(p, k_cache, v_cache, k_scale, v_scale, block_tables, bt_stride,
                     max_blocks_per_seq, context_lens, num_kv_heads, block_size, num_blocks, keys,
                     vals);
  if (st != NIA_OK) return st;
  p.tok = tok;
  p.head = head_dim;
  p.seq = tok * rows;
  p.k_start = k_start;
  p.k_len = k_len;
  p.start = rows;
  st = launch_gather(p, num_seqs, (hipStream_t)stream);
  if (st != NIA_OK) return st;
  return nia_prefill_split(out, out_tok_stride, out_head_stride, q, q_tok_stride, q_head_stride,
                           keys, tok, head_dim, vals, tok, head_dim, q_start, q_len, k_start, k_len,
                           num_seqs, max_q_len, num_heads, num_kv_heads, head_dim, scale, causal,
                           NIA_DTYPE_BF16, rows, split, split_bytes, stream);
}
