// stack_conv.h — the causal depth-wise convolutions in front of the layered designs' recurrences over long portions: conv_silu_kernel (stack_ssm.h) and delta_prep_kernel (stack_rec.h)
// with eight tokens of four channels a lane.
// What bounds them: their bytes, a row read and one written.  A token or a channel a thread, as those kernels have it for short portions, waits for a token's place in its entry and for its
// rows at every turn.  Here a wave asks for the rows of eight tokens and the taps - 1 before them at once; the few tiles at an entry's ends take what is not among them from the slot's tails.
// us: 2048 tokens of a delta rule's 4096 channels 89 -> 20 (67 MB), 10917 tokens of 4096 and 4608 channels 135 -> 88 and 146 -> 88 (358 and 402 MB; the silu's exponentials lie beside the bytes).
// The sums are those kernels', term by term and in their order, a head's sum of squares too (head_squares): a model answers with the same bits whichever form its steps take.
#pragma once
#include "stack_rec.h"
#include "stack_ssm.h"

namespace tgx {

constexpr int CONV_TOK = 8, CONV_WG_TOK = 4 * CONV_TOK, CONV_WG_CH = 256;      // tokens of a wave, of a workgroup; channels of both
// filtered[u] of tokens t0 + u (u < n): bias + sum over taps; the entry's tails kept.  raw: the projections' column of channel c; w[j]: tap j of four channels (the last: the current token's)
template <int TAPS>
__device__ __forceinline__ void conv_tile(const StepMeta& m, const float* raw, long long ldp, const f32x4* w, f32x4 b, float* state, size_t state_buf, int C, int c, int t0, int n, f32x4* filtered) {
  constexpr int NB = TAPS - 1;
  auto row = [&](int t) -> f32x4 { return *reinterpret_cast<const f32x4*>(raw + (long long)t * ldp); };
  auto fma4 = [](f32x4 x, f32x4 y, f32x4 z) { f32x4 o; for (int k = 0; k < 4; k++) o[k] = fmaf(x[k], y[k], z[k]); return o; };
  f32x4 x[CONV_TOK + NB];      // (rows outside the tile's own entry or behind the step's end are read and not used)
#pragma unroll
  for (int u = 0; u < CONV_TOK + NB; u++) x[u] = row(min(max(t0 - NB + u, 0), m.T - 1));
  const int i0 = m.tok_idx[t0], il = m.tok_idx[t0 + n - 1], cnt0 = m.tok_cnt[t0];
  if (n == CONV_TOK && il - i0 == CONV_TOK - 1 && i0 >= NB && cnt0 - il > NB) {      // (indices count on inside an entry only)
#pragma unroll
    for (int u = 0; u < CONV_TOK; u++) {
      f32x4 acc = b;
#pragma unroll
      for (int d = 0; d < TAPS; d++) acc = fma4(w[NB - d], x[u + NB - d], acc);
      filtered[u] = acc;
    }
    return;
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < CONV_TOK; u++) {
    if (u >= n) break;
    const int t = t0 + u, i = m.tok_idx[t], cnt = m.tok_cnt[t];
    const bool first = i < NB, last = cnt - i <= NB;
    const f32x4 x0 = x[u + NB];
    f32x4 acc = fma4(w[NB], x0, b);
    if (!first && !last) {
#pragma unroll
      for (int d = 1; d < TAPS; d++) acc = fma4(w[NB - d], x[u + NB - d], acc);
      filtered[u] = acc;
      continue;
    }
    const int pos = m.tok_pos[t], par = m.tok_par[t];
    const size_t srow = (size_t)m.tok_row[t] * NB * C + c;
    const float* st_old = state ? state + (size_t)par * state_buf + srow : nullptr;
    float* st_new = state ? state + (size_t)(par ^ 1) * state_buf + srow : nullptr;
#pragma unroll
    for (int d = 1; d < TAPS; d++) {
      f32x4 xv = x[u + NB - d];
      if (d > i) xv = pos - d >= 0 ? *reinterpret_cast<const f32x4*>(st_old + (size_t)(NB - (d - i)) * C) : zero;      // tail slot s holds position past - nb + s, past = pos - i
      acc = fma4(w[NB - d], xv, acc);
    }
    filtered[u] = acc;
    if (st_new) {
      const int s = NB - (cnt - i);                        // row i of cnt lands in tail slot nb - (cnt - i) ...
      if (s >= 0) *reinterpret_cast<f32x4*>(st_new + (size_t)s * C) = x0;
      if (i == 0)                                          // ... and an entry shorter than the tails keeps the end of the old ones
        for (int k = 0; k + cnt < NB; k++) *reinterpret_cast<f32x4*>(st_new + (size_t)k * C) = (pos - (NB - cnt - k) >= 0) ? *reinterpret_cast<const f32x4*>(st_old + (size_t)(k + cnt) * C) : zero;
    }
  }
}
template <int TAPS>
__device__ __forceinline__ void conv_taps(const float* cw, int c, f32x4* w) {      // [C][taps] -> per tap, four channels
  float v[4 * TAPS];
#pragma unroll
  for (int k = 0; k < TAPS; k++) { const f32x4 q = *reinterpret_cast<const f32x4*>(cw + (size_t)c * TAPS + 4 * k); for (int e = 0; e < 4; e++) v[4 * k + e] = q[e]; }
#pragma unroll
  for (int j = 0; j < TAPS; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) w[j][e] = v[e * TAPS + j];
}
__device__ __forceinline__ f32x4 silu4(f32x4 v) { f32x4 o; for (int k = 0; k < 4; k++) o[k] = silu_f(v[k]); return o; }

// Grid: (tokens / 32, C / 256 (+ 1 for the step sizes)); rows, channels and columns in fours
template <int TAPS>
__global__ __launch_bounds__(256) void conv_silu_tiles_kernel(StepMeta m, ConvSiluArgs a) {
  const int g0 = blockIdx.x * CONV_WG_TOK, g1 = min(m.T, g0 + CONV_WG_TOK);
  if (a.heads > 0 && blockIdx.y == gridDim.y - 1) {
    for (int i = threadIdx.x; i < (g1 - g0) * a.heads; i += 256) {
      const int t = g0 + i / a.heads, h = i % a.heads;
      const float dt = softplus_f(a.proj[(size_t)t * a.ldp + a.dt_col + h] + a.dt_bias[h]), la = -expf(a.a_log[h]) * dt;
      float* o = a.out + (size_t)t * a.ldo + a.C;
      o[h] = dt; o[a.heads + h] = expf(la); o[2 * a.heads + h] = la;
    }
    return;
  }
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t0 = g0 + CONV_TOK * wv, n = min(CONV_TOK, g1 - t0), c = blockIdx.y * CONV_WG_CH + 4 * lane;
  if (n <= 0 || c >= a.C) return;
  f32x4 w[TAPS], f[CONV_TOK];
  conv_taps<TAPS>(a.cw, c, w);
  conv_tile<TAPS>(m, a.proj + a.col0 + c, a.ldp, w, *reinterpret_cast<const f32x4*>(a.cb + c), a.state, a.state_buf, a.C, c, t0, n, f);
#pragma unroll
  for (int u = 0; u < CONV_TOK; u++) {
    if (u >= n) break;
    const f32x4 v = silu4(f[u]);
    *reinterpret_cast<f32x4*>(a.out + (size_t)(t0 + u) * a.ldo + c) = v;
    if (a.terms.out) store_terms4(a.terms, t0 + u, c, a.C, v);
  }
}

__device__ __forceinline__ float lane_xor4(float v) {      // the lane 4 apart: row_shl:4 for the even banks of four lanes, row_shr:4 for the odd ones
  const int b = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_amdgcn_update_dpp(0, b, 0x104, 0xf, 0x5, false), b, 0x114, 0xf, 0xa, false));
}
// the sum of a head's squares in the order of delta_prep_kernel, which has a channel a lane: over the channels 32 apart (the lower one's square is
// added unrounded to the upper one's), 16, 8 and 4 apart, which are here lanes, 2 and 1 apart, which are a lane's components, and 64 apart.  Every lane of the head gets it.  (A sum in another order moves the
// unit vectors in their last bits, which is enough to send a token with a near tie to another expert some layers on.)
template <int LPH>
__device__ __forceinline__ float head_squares(f32x4 v) {
#pragma clang fp contract(off)
  const bool upper = (threadIdx.x & 8) != 0;
  float s[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const float x = v[k];
    float y;
    if constexpr (LPH >= 16) {
      const float other = dpp_mov<0x128, 0xf>(x);          // row_ror:8: the lane 8 apart
      const float lo = upper ? other : x, hi = upper ? x : other;
      y = fmaf(lo, lo, hi * hi);
    } else y = x * x;
    y += lane_xor4(y);
    y += dpp_mov<0x4E, 0xf>(y);
    y += dpp_mov<0xB1, 0xf>(y);
    s[k] = y;
  }
  float ss = (s[0] + s[2]) + (s[1] + s[3]);
  if constexpr (LPH == 32) {
    const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(__float_as_uint(ss), __float_as_uint(ss), false, false));
    ss = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return ss;
}
// LPH: lanes of a q or k head (dim / 4).  Grid: (tokens / 32, C / 256 + 1 for the heads' gates)
template <int TAPS, int LPH>
__global__ __launch_bounds__(256) void delta_prep_tiles_kernel(StepMeta m, DeltaPrepArgs a) {
  const int g0 = blockIdx.x * CONV_WG_TOK, g1 = min(m.T, g0 + CONV_WG_TOK), GD = a.kv_heads * a.dim, C = 2 * GD + a.heads * a.vdim;
  if (blockIdx.y == gridDim.y - 1) {
    for (int i = threadIdx.x; i < (g1 - g0) * a.heads; i += 256) {
      const int t = g0 + i / a.heads, h = i % a.heads;
      const float* pr = a.proj + (size_t)t * a.ldp + a.col0;
      float* o = a.out + (size_t)t * a.ldo + C;
      o[h] = 1.0f / (1.0f + expf(-pr[a.b_col + h]));
      if (!a.a_log) continue;
      o[a.heads + h] = expf(-expf(a.a_log[h]) * softplus_f(pr[a.b_col + a.heads + h] + a.dt_bias[h]));
    }
    return;
  }
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t0 = g0 + CONV_TOK * wv, n = min(CONV_TOK, g1 - t0), c = blockIdx.y * CONV_WG_CH + 4 * lane;
  if (n <= 0 || c >= C) return;      // (a head's lanes leave together: C is whole heads of q and k, and the values are none)
  f32x4 w[TAPS], f[CONV_TOK];
  conv_taps<TAPS>(a.cw, c, w);
  conv_tile<TAPS>(m, a.proj + a.col0 + c, a.ldp, w, f32x4{0.f, 0.f, 0.f, 0.f}, a.state, a.state_buf, C, c, t0, n, f);
  const bool qk = c < 2 * GD, any_qk = (int)blockIdx.y * CONV_WG_CH < 2 * GD;
  const float scale = c < GD ? a.q_scale : 1.0f;
#pragma unroll
  for (int u = 0; u < CONV_TOK; u++) {
    if (u >= n) break;
    f32x4 v = silu4(f[u]);
    if (any_qk) {
      const float ss = head_squares<LPH>(v);      // (of value channels: not used)
      if (qk) v *= scale / sqrtf(ss + a.unit_eps);
    }
    *reinterpret_cast<f32x4*>(a.out + (size_t)(t0 + u) * a.ldo + c) = v;
  }
}

}  // namespace tgx
