// Fused QK-RMSNorm + RoPE / mRoPE + KV-cache write: the step that feeds the attention
// path (src/nano_inference/layers/attention.py:254-278), in one launch instead of the
// ~30 elementwise launches the PyTorch form takes per layer.
//
// Bound by HBM: q, k and v in, q, k and the cache rows out.  One wave takes 8-row groups
// of one token (its query heads, then its key heads); within a group 8 lanes share a row,
// lane c of the 8 holding dims 8 c .. + 7 and 64 + 8 c .. + 7, which are the pairs
// rotate_half combines: 16-byte accesses (each half of a row is one 128-byte line), no
// lane exchange in RoPE, three DPP steps for RMSNorm's sum.  The wave computes the
// token's 64 cosines and sines once, one frequency a lane, and every row of the token
// uses them from registers (a row a wave, 2-byte accesses and a sine and cosine per row
// before: 125 us at 8192 tokens of 32 + 8 heads in bf16, 1.75 TB/s; now 48-50 us, 4.4-4.5
// TB/s, where a large device copy reaches 5.0; 1000 tokens 16.4 -> 9.4 us; an fp8 cache at
// 4000 tokens of 28 + 4 heads 61 -> 18 us).  A token's rows may be spread over several waves
// (kRowsFillWaves), each with its own sines.  Measured and not taken: no prefetch of the next
// group (6 instead of 5 waves per SIMD, +-2%), 72 registers for 7 waves (spills, 77 us).
//
// Few rows (kFewRows; every decode step): qk_norm_rope_row_kernel, a wave per row, lane l holding
// dims l and l + 64.  All rows fit the chip at once, so the call takes one wave's time, and 16
// elements a lane take longer than two: 64 tokens of 28 + 4 heads 3.9 us in groups, 3.2 by rows;
// over an fp8 cache, where every element is divided by its row's scale, 5.3 and 3.7.
//
// Every rounding point of the PyTorch form is kept (T = the model dtype):
//   RMSNorm (src/nano_inference/layers/norm.py:35-47):
//     y = T( T( x * rsqrt(mean(x^2) + eps) ) * w )        mean and rsqrt in fp32
//   RoPE (src/nano_inference/layers/rotary.py:8-33, :104-130; mRoPE :184-210):
//     f = float(pos) * inv_freq[i],  c = T(cos f),  s = T(sin f)
//     out[d]      = T( T(y[d] * c)      + T(-y[d + 64] * s) )
//     out[d + 64] = T( T(y[d + 64] * c) + T(y[d] * s) )
//   with i = d for d < 64 (the table is cat(freqs, freqs)); for mRoPE the position
//   of frequency i comes from axis 0 (i < s0), 1 (i < s0 + s1) or 2.
// The mean's summation order differs from the PyTorch reduction, so a value lying on
// a rounding boundary can differ in its last bit; everything else is identical.
// With fp8 caches the rotated k row and the v row are stored as e4m3 codes with one
// fp32 scale per row (max |x| / 448), as nia_kv_write_fp8 stores them.
#include "common.h"
#include "work_map.h"

namespace {

struct RopeParams {
  void* q;
  int64_t q_tok, q_head;
  void* k;
  int64_t k_tok, k_head;
  const void* v;
  int64_t v_tok, v_head;
  const void* q_w;  // RMSNorm weights (model dtype) or null: no QK norm
  const void* k_w;
  float eps;
  const int64_t* pos;  // [num_axes][num_tokens] with axis stride pos_axis
  int64_t pos_axis;
  int32_t num_axes;    // 1 (RoPE) or 3 (mRoPE)
  const float* inv_freq;
  int32_t sec0, sec1;  // mRoPE: frequencies of the temporal and height axes
  void* k_cache;       // one layer [num_blocks][H_kv][BS][128], or null: no write
  void* v_cache;
  float* k_scale;      // fp8 caches: one scale per row, [num_blocks][H_kv][BS]
  float* v_scale;
  const int64_t* slots;
  int64_t num_slots;
  int32_t num_tokens, num_heads, num_kv_heads, block_size;
  int32_t parts, part_rows;  // waves per token, and the rows of each (a multiple of 8)
};

template <typename T>
struct Num;

template <>
struct Num<bf16_t> {
  static NIA_DEVICE float f(bf16_t x) { return (float)x; }
  static NIA_DEVICE bf16_t t(float x) { return (bf16_t)x; }  // round to nearest even
};

template <>
struct Num<float> {
  static NIA_DEVICE float f(float x) { return x; }
  static NIA_DEVICE float t(float x) { return x; }
};

constexpr int kRopeWaves = 4;  // waves per workgroup
// Rows up to which the call takes a wave per row.  By rows and in groups, us, bf16 / fp8 cache:
// 3200 rows 4.0 / 4.7 and 4.0 / 5.2, 4800 4.2 / 4.7 and 4.0 / 5.2, 6400 5.2 / 6.6 and 4.0 / 5.4.
// Over an fp8 cache also where a token's rows do not fill a group (4 + 1 heads, 2100 tokens: 7.1
// and 13.0): all lanes wait for the few that divide.
constexpr int64_t kFewRows = 5120;
constexpr int kRowGroup = 8;   // rows a wave handles at once (8 lanes each)
constexpr int kHalf = 8;       // dims per lane and row half
// Waves below which a token's row groups are spread over several waves (two per SIMD:
// every wave repeats the token's sines, so a fuller chip does not want more; aiming at
// 16384 waves gains 5% at 8192 tokens but costs 12-18% at 3000-4000).
constexpr int64_t kRowsFillWaves = 2048;

// Maximum over aligned groups of 8 lanes.
NIA_DEVICE float octet_max(float x) {
  x = fmaxf(x, dpp_f32<kDppQuadXor1>(x));
  x = fmaxf(x, dpp_f32<kDppQuadXor2>(x));
  return fmaxf(x, dpp_f32<kDppRowHalfMirror>(x));
}

// Eight consecutive elements.  VEC: 16-byte accesses (pointers and strides checked on the
// host), else element by element.
template <typename T>
using Vec8 = T __attribute__((ext_vector_type(kHalf)));

template <typename T, bool VEC>
NIA_DEVICE Vec8<T> load8(const T* p) {
  typedef T Chunk __attribute__((ext_vector_type(16 / sizeof(T))));
  Vec8<T> r;
  if constexpr (VEC && sizeof(T) == 2) {
    r = *reinterpret_cast<const Chunk*>(p);
  } else if constexpr (VEC) {
    const Chunk a = reinterpret_cast<const Chunk*>(p)[0], b = reinterpret_cast<const Chunk*>(p)[1];
    r = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
  } else {
#pragma unroll
    for (int i = 0; i < kHalf; ++i) r[i] = p[i];
  }
  return r;
}

template <typename T, bool VEC>
NIA_DEVICE void store8(T* p, const Vec8<T>& r) {
  typedef T Chunk __attribute__((ext_vector_type(16 / sizeof(T))));
  if constexpr (VEC && sizeof(T) == 2) {
    *reinterpret_cast<Chunk*>(p) = r;
  } else if constexpr (VEC) {
    reinterpret_cast<Chunk*>(p)[0] = __builtin_shufflevector(r, r, 0, 1, 2, 3);
    reinterpret_cast<Chunk*>(p)[1] = __builtin_shufflevector(r, r, 4, 5, 6, 7);
  } else {
#pragma unroll
    for (int i = 0; i < kHalf; ++i) p[i] = r[i];
  }
}

// Eight e4m3 codes of x for a row scale (zero row: scale 0, codes 0).
template <typename T, bool VEC>
NIA_DEVICE void store_codes(uint8_t* p, const Vec8<T>& x, float scale) {
  uint32_t w[2] = {0u, 0u};
  if (scale > 0.f) {
#pragma unroll
    for (int i = 0; i < kHalf; i += 2)
      w[i >> 2] |= fp8x2_from_f32(Num<T>::f(x[i]) / scale, Num<T>::f(x[i + 1]) / scale)
                   << (8 * (i & 2));
  }
  if constexpr (VEC) {
    *reinterpret_cast<uint2*>(p) = make_uint2(w[0], w[1]);
  } else {
#pragma unroll
    for (int i = 0; i < kHalf; ++i) p[i] = (uint8_t)(w[i >> 2] >> (8 * (i & 3)));
  }
}

// Largest magnitude of a row's elements; NaN elements are left out, but a row of nothing else
// keeps NaN (starting from 0 would turn it into a row of zeros).
template <typename T>
NIA_DEVICE float octet_amax(const Vec8<T>& a, const Vec8<T>& b) {
  float m = fmaxf(fabsf(Num<T>::f(a[0])), fabsf(Num<T>::f(b[0])));
#pragma unroll
  for (int i = 1; i < kHalf; ++i)
    m = fmaxf(m, fmaxf(fabsf(Num<T>::f(a[i])), fabsf(Num<T>::f(b[i]))));
  return octet_max(m);
}

// FP8: the caches hold e4m3 codes with one fp32 scale per row, max |x| / 448.
template <typename T, bool FP8, bool VEC>
__global__ __launch_bounds__(kRopeWaves * kWave) void qk_norm_rope_kernel(RopeParams p) {
  using N = Num<T>;
  constexpr int D = 128;
  const int lane = threadIdx.x & (kWave - 1);
  // parts exceeds 1 only for few tokens, so the wave number fits 32 bits
  const uint32_t w = blockIdx.x * kRopeWaves + (uint32_t)uniform(threadIdx.x >> 6);
  const int64_t tok = p.parts == 1 ? w : w / (uint32_t)p.parts;
  const int part = (int)(w - (uint32_t)tok * (uint32_t)p.parts);
  if (tok >= p.num_tokens) return;
  const int rows = p.num_heads + p.num_kv_heads;
  const int r_end = min(rows, (part + 1) * p.part_rows);
  const int sub = lane >> 3;        // row of the group
  const int d0 = kHalf * (lane & 7);  // the lane's dims d0 .. + 7 and 64 + d0 .. + 7

  // A row group's rows, loaded together: this lane's halves of x, and of v for key rows.
  struct Row {
    Vec8<T> lo, hi, vlo, vhi;
    T* x;
    int hk;   // key head, negative for query heads
    bool ok;
  };
  // the cache row of the token's slot for KV head 0, or -1: nothing is written
  int64_t cache_row = -1;
  if (p.k_cache != nullptr) {
    const int64_t slot = p.slots[tok];
    if (slot >= 0 && slot < p.num_slots) {
      const int64_t blk = slot / p.block_size;
      cache_row = blk * p.num_kv_heads * p.block_size + (slot - blk * p.block_size);
    }
  }
  auto load_rows = [&](int r0, Row& y) __attribute__((always_inline)) {
    const int r = r0 + sub;
    y.ok = r < r_end;
    y.hk = r - p.num_heads;
    if (!y.ok) return;
    y.x = y.hk < 0 ? reinterpret_cast<T*>(p.q) + tok * p.q_tok + (int64_t)r * p.q_head
                   : reinterpret_cast<T*>(p.k) + tok * p.k_tok + (int64_t)y.hk * p.k_head;
    y.lo = load8<T, VEC>(y.x + d0);
    y.hi = load8<T, VEC>(y.x + 64 + d0);
    if (y.hk >= 0 && cache_row >= 0) {
      const T* vr = reinterpret_cast<const T*>(p.v) + tok * p.v_tok + (int64_t)y.hk * p.v_head;
      y.vlo = load8<T, VEC>(vr + d0);
      y.vhi = load8<T, VEC>(vr + 64 + d0);
    }
  };

  Row cur;
  load_rows(part * p.part_rows, cur);  // in flight while the sines are computed
  float c[kHalf], s[kHalf];
  {
    const int axis =
        p.num_axes == 1 ? 0 : (lane < p.sec0 ? 0 : (lane < p.sec0 + p.sec1 ? 1 : 2));
    const float ang = (float)p.pos[axis * p.pos_axis + tok] * p.inv_freq[lane];
    const float cl = N::f(N::t(cosf(ang)));
    const float sl = N::f(N::t(sinf(ang)));
#pragma unroll
    for (int i = 0; i < kHalf; ++i) {
      c[i] = __shfl(cl, d0 + i, kWave);
      s[i] = __shfl(sl, d0 + i, kWave);
    }
  }

  for (int r0 = part * p.part_rows; r0 < r_end; r0 += kRowGroup) {
    Row nxt;
    nxt.ok = false;
    if (r0 + kRowGroup < r_end) load_rows(r0 + kRowGroup, nxt);
    if (cur.ok) {
      const T* wt = reinterpret_cast<const T*>(cur.hk < 0 ? p.q_w : p.k_w);
      float y0[kHalf], y1[kHalf];
#pragma unroll
      for (int i = 0; i < kHalf; ++i) {
        y0[i] = N::f(cur.lo[i]);
        y1[i] = N::f(cur.hi[i]);
      }
      if (wt != nullptr) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < kHalf; ++i) ss += y0[i] * y0[i] + y1[i] * y1[i];
        ss = group_sum<8>(ss);
        const float r = rsqrtf(ss / (float)D + p.eps);
        const Vec8<T> w0 = load8<T, VEC>(wt + d0), w1 = load8<T, VEC>(wt + 64 + d0);
#pragma unroll
        for (int i = 0; i < kHalf; ++i) {
          y0[i] = N::f(N::t(N::f(N::t(y0[i] * r)) * N::f(w0[i])));
          y1[i] = N::f(N::t(N::f(N::t(y1[i] * r)) * N::f(w1[i])));
        }
      }
      Vec8<T> o0, o1;
#pragma unroll
      for (int i = 0; i < kHalf; ++i) {
        o0[i] = N::t(N::f(N::t(y0[i] * c[i])) + N::f(N::t(-y1[i] * s[i])));
        o1[i] = N::t(N::f(N::t(y1[i] * c[i])) + N::f(N::t(y0[i] * s[i])));
      }
      store8<T, VEC>(cur.x + d0, o0);
      store8<T, VEC>(cur.x + 64 + d0, o1);
      if (cur.hk >= 0 && cache_row >= 0) {
        const int64_t row = cache_row + (int64_t)cur.hk * p.block_size;
        if constexpr (FP8) {
          const float ks = octet_amax<T>(o0, o1) / kE4m3Max;
          const float vs = octet_amax<T>(cur.vlo, cur.vhi) / kE4m3Max;
          uint8_t* kc = reinterpret_cast<uint8_t*>(p.k_cache) + row * D + d0;
          uint8_t* vc = reinterpret_cast<uint8_t*>(p.v_cache) + row * D + d0;
          store_codes<T, VEC>(kc, o0, ks);
          store_codes<T, VEC>(kc + 64, o1, ks);
          store_codes<T, VEC>(vc, cur.vlo, vs);
          store_codes<T, VEC>(vc + 64, cur.vhi, vs);
          if ((lane & 7) == 0) {
            p.k_scale[row] = ks;
            p.v_scale[row] = vs;
          }
        } else {
          T* kc = reinterpret_cast<T*>(p.k_cache) + row * D + d0;
          T* vc = reinterpret_cast<T*>(p.v_cache) + row * D + d0;
          store8<T, VEC>(kc, o0);
          store8<T, VEC>(kc + 64, o1);
          store8<T, VEC>(vc, cur.vlo);
          store8<T, VEC>(vc + 64, cur.vhi);
        }
      }
    }
    cur = nxt;
  }
}

// Row maximum of |x| over the wave's 128 values (two per lane); NaN as in octet_amax.
NIA_DEVICE float row_amax(float a, float b) {
  float m = fmaxf(fabsf(a), fabsf(b));
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) m = fmaxf(m, __shfl_xor(m, off, kWave));
  return m;
}

// e4m3 code of x for a row scale (zero row: scale 0, code 0).
NIA_DEVICE uint8_t fp8_code(float x, float scale) {
  return scale > 0.f ? (uint8_t)(fp8x2_from_f32(x / scale, 0.f) & 0xffu) : (uint8_t)0;
}

// One wave per (token, head) row: rows 0 .. H - 1 of a token are its query heads, the others its
// key heads.
template <typename T, bool FP8>
__global__ __launch_bounds__(kRopeWaves * kWave) void qk_norm_rope_row_kernel(RopeParams p) {
  using N = Num<T>;
  constexpr int D = 128;
  const int lane = threadIdx.x & (kWave - 1);
  const int per_tok = p.num_heads + p.num_kv_heads;
  const int64_t row = (int64_t)blockIdx.x * kRopeWaves + (threadIdx.x >> 6);
  if (row >= (int64_t)p.num_tokens * per_tok) return;
  const int tok = (int)(row / per_tok);
  const int hh = (int)(row - (int64_t)tok * per_tok);
  const bool is_q = hh < p.num_heads;
  const int hk = hh - p.num_heads;
  T* x = is_q ? reinterpret_cast<T*>(p.q) + tok * p.q_tok + (int64_t)hh * p.q_head
              : reinterpret_cast<T*>(p.k) + tok * p.k_tok + (int64_t)hk * p.k_head;
  const T* w = reinterpret_cast<const T*>(is_q ? p.q_w : p.k_w);

  float y0 = N::f(x[lane]);
  float y1 = N::f(x[lane + 64]);
  if (w != nullptr) {
    float ss = y0 * y0 + y1 * y1;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) ss += __shfl_xor(ss, off, kWave);
    const float r = rsqrtf(ss / (float)D + p.eps);
    y0 = N::f(N::t(N::f(N::t(y0 * r)) * N::f(w[lane])));
    y1 = N::f(N::t(N::f(N::t(y1 * r)) * N::f(w[lane + 64])));
  }
  const int axis = p.num_axes == 1 ? 0 : (lane < p.sec0 ? 0 : (lane < p.sec0 + p.sec1 ? 1 : 2));
  const float ang = (float)p.pos[axis * p.pos_axis + tok] * p.inv_freq[lane];
  const float c = N::f(N::t(cosf(ang)));
  const float s = N::f(N::t(sinf(ang)));
  const T o0 = N::t(N::f(N::t(y0 * c)) + N::f(N::t(-y1 * s)));
  const T o1 = N::t(N::f(N::t(y1 * c)) + N::f(N::t(y0 * s)));
  x[lane] = o0;
  x[lane + 64] = o1;
  if (is_q || p.k_cache == nullptr) return;
  const int64_t slot = p.slots[tok];
  if (slot < 0 || slot >= p.num_slots) return;
  const int64_t blk = slot / p.block_size;
  const int64_t cache_row =
      (blk * p.num_kv_heads + hk) * p.block_size + (slot - blk * p.block_size);
  const T* vr = reinterpret_cast<const T*>(p.v) + tok * p.v_tok + (int64_t)hk * p.v_head;
  const T v0 = vr[lane], v1 = vr[lane + 64];
  if constexpr (FP8) {
    const float ks = row_amax(N::f(o0), N::f(o1)) / kE4m3Max;
    const float vs = row_amax(N::f(v0), N::f(v1)) / kE4m3Max;
    uint8_t* kc = reinterpret_cast<uint8_t*>(p.k_cache) + cache_row * D + lane;
    uint8_t* vc = reinterpret_cast<uint8_t*>(p.v_cache) + cache_row * D + lane;
    kc[0] = fp8_code(N::f(o0), ks);
    kc[64] = fp8_code(N::f(o1), ks);
    vc[0] = fp8_code(N::f(v0), vs);
    vc[64] = fp8_code(N::f(v1), vs);
    if (lane == 0) {
      p.k_scale[cache_row] = ks;
      p.v_scale[cache_row] = vs;
    }
  } else {
    T* kc = reinterpret_cast<T*>(p.k_cache) + cache_row * D + lane;
    T* vc = reinterpret_cast<T*>(p.v_cache) + cache_row * D + lane;
    kc[0] = o0;
    kc[64] = o1;
    vc[0] = v0;
    vc[64] = v1;
  }
}

// 16-byte accesses: aligned pointers, strides of whole 16-byte groups.
bool rope_vec_ok(const RopeParams& p, int es, bool write, bool fp8) {
  auto ptr = [](const void* x, int a) { return (uintptr_t)x % a == 0; };
  auto st = [&](int64_t x) { return x * es % 16 == 0; };
  if (!ptr(p.q, 16) || !st(p.q_tok) || !st(p.q_head) || !ptr(p.k, 16) || !st(p.k_tok) ||
      !st(p.k_head) || !ptr(p.q_w, 16) || !ptr(p.k_w, 16))
    return false;
  if (!write) return true;
  const int ca = fp8 ? 8 : 16;
  return ptr(p.v, 16) && st(p.v_tok) && st(p.v_head) && ptr(p.k_cache, ca) && ptr(p.v_cache, ca);
}

template <typename T, bool FP8>
void launch_rope(const RopeParams& p, dim3 grid, bool by_rows, bool vec, hipStream_t s) {
  const dim3 block(kRopeWaves * kWave);
  if (by_rows)
    nia_launch((qk_norm_rope_row_kernel<T, FP8>), grid, block, s, p);
  else if (vec)
    nia_launch((qk_norm_rope_kernel<T, FP8, true>), grid, block, s, p);
  else
    nia_launch((qk_norm_rope_kernel<T, FP8, false>), grid, block, s, p);
}

}  // namespace

namespace {

int32_t launch_qk_norm_rope(
    void* q, int64_t q_tok_stride, int64_t q_head_stride, void* k, int64_t k_tok_stride,
    int64_t k_head_stride, const void* v, int64_t v_tok_stride, int64_t v_head_stride,
    const void* q_norm_weight, const void* k_norm_weight, float eps, const int64_t* positions,
    int64_t pos_axis_stride, int32_t num_axes, const float* inv_freq, int32_t mrope_section0,
    int32_t mrope_section1, void* k_cache, void* v_cache, float* k_scale, float* v_scale,
    bool fp8, const int64_t* slot_mapping, int32_t num_tokens, int32_t num_heads,
    int32_t num_kv_heads, int32_t head_dim, int32_t block_size, int64_t num_blocks,
    int32_t dtype, void* stream) {
  if (num_tokens < 0 || num_heads < 0 || num_kv_heads < 0) return NIA_ERR_INVALID_ARGUMENT;
  if (num_axes != 1 && num_axes != 3) return NIA_ERR_INVALID_ARGUMENT;
  if (num_axes == 3 && (mrope_section0 < 0 || mrope_section1 < 0 ||
                        mrope_section0 + mrope_section1 > head_dim / 2))
    return NIA_ERR_INVALID_ARGUMENT;
  if ((q_norm_weight != nullptr || k_norm_weight != nullptr) && !(eps >= 0.f))
    return NIA_ERR_INVALID_ARGUMENT;
  if (num_tokens == 0 || num_heads + num_kv_heads == 0) return NIA_OK;
  if ((num_heads > 0 && !q) || (num_kv_heads > 0 && !k) || !positions || !inv_freq)
    return NIA_ERR_INVALID_ARGUMENT;
  const bool write = k_cache != nullptr;
  if (write && (!v_cache || !v || !slot_mapping || block_size <= 0 || num_blocks < 0 ||
                num_kv_heads == 0))
    return NIA_ERR_INVALID_ARGUMENT;
  if (fp8 && (!write || !k_scale || !v_scale)) return NIA_ERR_INVALID_ARGUMENT;
  if (head_dim != 128 || (dtype != NIA_DTYPE_BF16 && dtype != NIA_DTYPE_F32))
    return NIA_ERR_UNSUPPORTED;
  const int64_t rows = (int64_t)num_heads + num_kv_heads;
  RopeParams p{};
  p.q = q;
  p.q_tok = q_tok_stride;
  p.q_head = q_head_stride;
  p.k = k;
  p.k_tok = k_tok_stride;
  p.k_head = k_head_stride;
  p.v = v;
  p.v_tok = v_tok_stride;
  p.v_head = v_head_stride;
  p.q_w = q_norm_weight;
  p.k_w = k_norm_weight;
  p.eps = eps;
  p.pos = positions;
  p.pos_axis = pos_axis_stride;
  p.num_axes = num_axes;
  p.inv_freq = inv_freq;
  p.sec0 = mrope_section0;
  p.sec1 = mrope_section1;
  p.k_cache = k_cache;
  p.v_cache = v_cache;
  p.k_scale = k_scale;
  p.v_scale = v_scale;
  p.slots = slot_mapping;
  p.num_slots = num_blocks * block_size;
  p.num_tokens = num_tokens;
  p.num_heads = num_heads;
  p.num_kv_heads = num_kv_heads;
  p.block_size = block_size;
  // A token's row groups over as many waves as it takes to fill the chip.
  const int64_t row_groups = (rows + kRowGroup - 1) / kRowGroup;
  int64_t parts = (kRowsFillWaves + num_tokens - 1) / num_tokens;
  if (parts > row_groups) parts = row_groups;
  const int64_t per_part = (row_groups + parts - 1) / parts;
  parts = (row_groups + per_part - 1) / per_part;  // no empty part
  p.parts = (int32_t)parts;
  p.part_rows = (int32_t)(per_part * kRowGroup);
  const bool by_rows = num_tokens * rows <= kFewRows || (fp8 && rows < kRowGroup);
  const int64_t wgs =
      ((int64_t)num_tokens * (by_rows ? rows : parts) + kRopeWaves - 1) / kRopeWaves;
  if (wgs > kMaxGroups) return NIA_ERR_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)wgs);
  const bool bf16 = dtype == NIA_DTYPE_BF16;
  const bool vec = rope_vec_ok(p, bf16 ? 2 : 4, write, fp8);
  if (bf16 && fp8)
    launch_rope<bf16_t, true>(p, grid, by_rows, vec, s);
  else if (bf16)
    launch_rope<bf16_t, false>(p, grid, by_rows, vec, s);
  else if (fp8)
    launch_rope<float, true>(p, grid, by_rows, vec, s);
  else
    launch_rope<float, false>(p, grid, by_rows, vec, s);
  return hipGetLastError() == hipSuccess ? NIA_OK : NIA_ERR_LAUNCH;
}

}  // namespace

extern "C" int32_t nia_qk_norm_rope_kv_write(
    void* q, int64_t q_tok_stride, int64_t q_head_stride, void* k, int64_t k_tok_stride,
    int64_t k_head_stride, const void* v, int64_t v_tok_stride, int64_t v_head_stride,
    const void* q_norm_weight, const void* k_norm_weight, float eps, const int64_t* positions,
    int64_t pos_axis_stride, int32_t num_axes, const float* inv_freq, int32_t mrope_section0,
    int32_t mrope_section1, void* k_cache, void* v_cache, const int64_t* slot_mapping,
    int32_t num_tokens, int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
    int32_t block_size, int64_t num_blocks, int32_t dtype, void* stream) {
  return launch_qk_norm_rope(q, q_tok_stride, q_head_stride, k, k_tok_stride, k_head_stride, v,
                             v_tok_stride, v_head_stride, q_norm_weight, k_norm_weight, eps,
                             positions, pos_axis_stride, num_axes, inv_freq, mrope_section0,
                             mrope_section1, k_cache, v_cache, nullptr, nullptr, false,
                             slot_mapping, num_tokens, num_heads, num_kv_heads, head_dim,
                             block_size, num_blocks, dtype, stream);
}

extern "C" int32_t nia_qk_norm_rope_kv_write_fp8(
    void* q, int64_t q_tok_stride, int64_t q_head_stride, void* k, int64_t k_tok_stride,
    int64_t k_head_stride, const void* v, int64_t v_tok_stride, int64_t v_head_stride,
    const void* q_norm_weight, const void* k_norm_weight, float eps, const int64_t* positions,
    int64_t pos_axis_stride, int32_t num_axes, const float* inv_freq, int32_t mrope_section0,
    int32_t mrope_section1, void* k_cache, void* v_cache, float* k_scale, float* v_scale,
    const int64_t* slot_mapping, int32_t num_tokens, int32_t num_heads, int32_t num_kv_heads,
    int32_t head_dim, int32_t block_size, int64_t num_blocks, int32_t dtype, void* stream) {
  return launch_qk_norm_rope(q, q_tok_stride, q_head_stride, k, k_tok_stride, k_head_stride, v,
                             v_tok_stride, v_head_stride, q_norm_weight, k_norm_weight, eps,
                             positions, pos_axis_stride, num_axes, inv_freq, mrope_section0,
                             mrope_section1, k_cache, v_cache, k_scale, v_scale, true,
                             slot_mapping, num_tokens, num_heads, num_kv_heads, head_dim,
                             block_size, num_blocks, dtype, stream);
}
