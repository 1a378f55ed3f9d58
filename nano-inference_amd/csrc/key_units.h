// Keys into cache blocks and units into ranges: plain integer code for the device and for the
// host (the launchers; tests compile it with the host's compiler).
#pragma once

#include <stdint.h>

#ifdef __HIP__
#define NIA_BOTH __host__ __device__ __forceinline__
#else
#define NIA_BOTH inline
#endif

// Division of 0 <= x < 2^31 by d >= 1 (a block size, a group) as mulhi(x, m) >> s: with
// l = ceil(log2 d) and m = ceil(2^(31 + l) / d) (< 2^32 since d > 2^(l - 1)), m d - 2^(31 + l)
// < d <= 2^l, so floor(x m / 2^(31 + l)) = floor(x / d) for every x < 2^31 (the round-up
// method of Granlund and Montgomery, "Division by invariant integers using
// multiplication", 1994).  For d = 2^k it is m = 2^31, s = k - 1: the shift by k.
inline void block_divisor(int32_t d, uint32_t& m, int32_t& s) {
  if (d <= 1) {  // no 32-bit m divides by 1: every key maps to block 0 (the kernels that
    m = 0;        // use this take block sizes >= 4; block size 1 is routed elsewhere)
    s = 0;
    return;
  }
  int l = 1;
  while ((int64_t)1 << l < d) ++l;
  m = (uint32_t)((((uint64_t)1 << (31 + l)) + (uint64_t)d - 1) / (uint64_t)d);
  s = l - 1;
}

// x / d under the divisor (m, s) of block_divisor.
NIA_BOTH int key_block(int x, uint32_t m, int s) {
  return (int)((uint32_t)((uint64_t)(uint32_t)x * m >> 32) >> s);
}

constexpr int kCombineRows = 16;  // partial rows a wave of the decode's merge takes at a time

// Few units (at most two per workgroup that has a CU to itself, `alone` ranges): one or two to a
// range, and only as many ranges as that takes.  Spread over every resident wave, a sequence's
// units would lie between empty ranges, which the merge walks as well: one sequence of 1023 keys
// (16 query, 8 KV heads) had 256 ranges to merge, 39.8 us; with one unit a range 10.3 us (two:
// 12.4, four: 16.4).  One sequence of 8192 keys (32 and 8 heads) 45.7 us before, 17.2 with one
// unit a range (two workgroups per CU), 15.3 with two, 17.7 with four.
NIA_BOTH bool few_units(int64_t total, int64_t alone) { return total <= 2 * alone; }

// Units a range, of `ranges` in all: two past `alone` (the merge is what they save), one where
// the `sequences` (sequence, KV head group) pairs are short enough for a merge in one round
// either way: 130 sequences of up to 141 keys (32 and 4 heads) 16.6 us with two, 15.3 with one.
NIA_BOTH int64_t few_units_a_range(int64_t total, int64_t alone, int64_t ranges,
                                   int64_t sequences) {
  return total <= alone || (total <= ranges && total <= kCombineRows * sequences) ? 1 : 2;
}

// Waves per (sequence, head) pair in the merge of a decode whose `ranges` hold `sequences`
// (sequence, KV head group) pairs.  Few pairs (a small batch, whose sequences lie in many ranges)
// leave the chip to it: with at most 256 pairs 16 waves each, at most 1024 four, i.e. at most
// 4096 waves (half of what the chip holds): a sequence of 8000 keys among 23 of 100 (32 and 8
// heads) 35 us with one wave a pair, 22 with four.  Four only where there are eight ranges a
// sequence or more: with fewer the other three waves find nothing to do and cost their launch
// (59 sequences of up to 238 keys, 16 and 8 heads, 13.7 us instead of 12.8).  The 2048 pairs of
// 64 sequences of 32 heads, each in few ranges, keep one wave (190 us either way).
inline int merge_waves(int64_t pairs, int64_t ranges, int64_t sequences) {
  if (pairs <= 256) return 16;
  return pairs <= 1024 && ranges >= 8 * sequences ? 4 : 1;
}
