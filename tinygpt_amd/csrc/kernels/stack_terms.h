// stack_terms.h — rows that a matrix-core product reads as lines of two 16-bit terms (stack_line.h), written by the kernel that makes them.
#pragma once
#include "common.h"

namespace tgx {

// Row t of W channels (a multiple of 32) at t * 2 W: [W / 32][32 first terms | 32 second terms].  In place of a launch that reads the rows and writes them again in front of the product
// (2048 rows of 2048 channels 8.4 us).
struct RowTerms { bf16_t* out; int half, one_term; };      // (half: fp16 terms; out nullptr: none)
__device__ __forceinline__ void term_pair(const RowTerms& a, float v, bf16_t& hi, bf16_t& lo) {
  if (a.half) split16<DT_F16>(v, hi, lo); else split16<DT_BF16>(v, hi, lo);
  if (a.one_term) lo = 0;
}
__device__ __forceinline__ bf16_t* term_line(const RowTerms& a, size_t t, int c, int W) { return a.out + t * 2 * W + (size_t)(c >> 5) * 64 + (c & 31); }
__device__ __forceinline__ void store_term(const RowTerms& a, size_t t, int c, int W, float v) {
  bf16_t* line = term_line(a, t, c, W);
  term_pair(a, v, line[0], line[32]);
}
__device__ __forceinline__ void store_terms4(const RowTerms& a, size_t t, int c, int W, f32x4 v) {      // c a multiple of four
  unsigned int h[2], l[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    bf16_t hi[2], lo[2];
#pragma unroll
    for (int u = 0; u < 2; u++) term_pair(a, v[2 * i + u], hi[u], lo[u]);
    h[i] = (unsigned int)hi[0] | ((unsigned int)hi[1] << 16);
    l[i] = (unsigned int)lo[0] | ((unsigned int)lo[1] << 16);
  }
  bf16_t* line = term_line(a, t, c, W);
  *reinterpret_cast<uint2*>(line) = uint2{h[0], h[1]};
  *reinterpret_cast<uint2*>(line + 32) = uint2{l[0], l[1]};
}

}  // namespace tgx
