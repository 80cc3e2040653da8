// stack_rec_block.h — the recurrences of stack_rec.h whose decay is a number per key channel or that correct what they store (REC_WKV, REC_DELTA, REC_CDELTA), over long portions,
// 32 tokens at a time on the fp32 matrix cores (v_mfma_f32_16x16x4_f32: nothing is rounded below fp32).
// With w_t the decays (a vector over the key channels; one number for all of them in REC_DELTA) and D(i, t) = w_(i+1) .. w_t, a block of 32 tokens on a state S unrolls to
//   delta:  u_t = beta_t (v_t - (k_t D(0, t))^T S) - sum_{i < t} A_ti u_i,  A_ti = beta_t sum_d k_t k_i D(i, t)      (the rows of a unit lower triangular system)
//           o_t = (q_t D(0, t))^T S + sum_{i <= t} P_ti u_i,                P_ti = sum_d q_t k_i D(i, t)
//   wkv:    u_t = v_t,  o_t = (r_t D(0, t - 1))^T S + sum_{i < t} (sum_d r_t k_i D(i, t - 1)) v_i + (sum_d r_t u k_t) v_t
//   S <- diag(D(0, 32)) S + sum_i (k_i D(i, 32)) u_i^T
//   rec_block_prep_kernel   what no state is needed for, every block of every head by itself: P, the decayed rows, and the system solved for its two right-hand sides, so that
//                           u = U - W S with U from beta v and W from beta k D
//   rec_block_kernel        one workgroup per (entry, head, 16 value channels) walks the entry's blocks: three products a block with the state in matrix-core accumulators
// Every D is a product of decays as they are: no logarithms, no quotients, so decays of zero and blocks whose whole product underflows are nothing special.  Blocks are counted from
// the entry's first token; a block past the entry's end is padded by tokens with q = k = v = beta = 0 and w = 1, which change nothing.
// A number that is not finite reaches the outputs of the earlier tokens of its block too (a factor of zero times it), as in the scalar-decay blocks and the matrix-core attentions; never another request.
//
// What bounds it: the token by token scan is a chain of one dependent read-update step a token, of one wave's instructions (0.13 to 0.17 us each); here the chain has a 32nd of the steps, of
// 1.7 us (delta rules of up to 128 key channels; of 64 1.1) and 1.1 us (wkv; 0.75).  A block's operands are 68 KB a workgroup (40 KB) and 52 KB (32 KB), as long in a compute unit's memory
// pipeline (delta, 128 channels: 1.3 us without the matrix instructions) as its matrix instructions beside them (1.5 us without the loads).  Blocks of 32: longer ones have as many bytes
// and products a token and twice the pairs.  2048 tokens, us, scan -> preparation + blocks: delta rule of 16 heads of 128 x 128 338 -> 48 + 109 (in a model's pass, its inputs not in the cache, 51 + 118),
// with a decay a channel (8 heads) 353 -> 30 + 106, wkv of 32 heads of 64 x 64 251 -> 45 + 48 (50 + 50).
#pragma once
#include <type_traits>

#include "common.h"
#include "stack_meta.h"
#include "stack_rec_args.h"

namespace tgx {

typedef __attribute__((ext_vector_type(2))) float f32x2;
// a (block, head)'s part of the scratch, in floats.  Q, K, W: the matrix cores' fragments [16-channel tile][16-token tile][lane][4] (Q, W: lane = 16 (d % 16 / 4) + t % 16, four
// channels; K: lane = 16 (t % 16 / 4) + d % 16, four tokens); U: [16-column tile][16-token tile][lane = 16 (t % 16 / 4) + e % 16][4 tokens]; P: [i % 4][lane = 16 (i % 16 / 4) + t % 16]
// [2 (t / 16) + i / 16]; G: D(0, 32) per channel
struct RecBlockLayout {
  int dp, ep;      // key channels in 64s, value channels in 16s
  int q, k, w, u, p, g, stride;
  __host__ __device__ RecBlockLayout(int dim, int vdim, bool solve) {
    dp = (dim + 63) / 64 * 64; ep = (vdim + 15) / 16 * 16;
    q = 0; k = REC_BLOCK * dp; w = 2 * REC_BLOCK * dp; u = w + (solve ? REC_BLOCK * dp : 0); p = u + REC_BLOCK * ep; g = p + REC_BLOCK * REC_BLOCK; stride = g + dp;
  }
};
// the first block of an entry in the scratch: entries never share a block
__host__ __device__ __forceinline__ int rec_first_block(int start, int e) { return start / REC_BLOCK + e; }

// the sum of a number over eight adjacent lanes in 64 bits
__device__ __forceinline__ double row_sum8(double v) {
  auto from = [&](auto C) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned int)b, decltype(C)::value, 0xf, 0xf, false), hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned int)(b >> 32), decltype(C)::value, 0xf, 0xf, false);
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
  };
  v += from(std::integral_constant<int, 0xB1>{});       // quad_perm:[1,0,3,2]
  v += from(std::integral_constant<int, 0x4E>{});       // quad_perm:[2,3,0,1]
  return v + from(std::integral_constant<int, 0x141>{});      // row_half_mirror
}

// Grid: (blocks of the longest entry, heads, entries).  DP: 64 or 128 key channels.
// The pairs: lane = (earlier token i, an eighth of the channels), r = k_i D(i, t) carried from t to t + 1, so a pair costs its products and one sum over eight lanes.  The system: a
// thread per column of either right-hand side, the 32 unknowns in registers, A's rows from LDS for all lanes at once.
// Rounding: a block's pairs enter 32 tokens' outputs and its decays all of the state, where the scan rounds each token's by itself, so the sum of a pair behind its sixteen chains of products
// and the products of decays run in 64 bits, and what the earlier tokens take from an equation is summed apart from its right-hand side.  Against 64 bits, operation by operation on a
// CPU (128 x 128, 320 tokens; outputs / state, the scan's error = 1): delta 1.55 / 1.7 without these, 1.00 / 0.9 with them, a decay a channel 1.4 / 1.4 and 0.95 / 0.8, wkv 1.06 / 1.1 and
// 0.88 / 1.0.
template <int KIND, int DP>
__global__ __launch_bounds__(256, KIND == REC_WKV ? 3 : 2) void rec_block_prep_kernel(StepMeta m, RecScanArgs a, float* scratch) {
  constexpr int Q = REC_BLOCK, R4 = DP / 4, DPT = DP / 8;      // floats in fours a row, channels per lane of a pair
  constexpr bool SCALAR = KIND == REC_DELTA, SOLVE = KIND != REC_WKV;
  __shared__ __attribute__((aligned(16))) float s_q[Q][DP], s_k[Q][DP], s_w[SCALAR ? 1 : Q][DP];
  __shared__ __attribute__((aligned(16))) float s_A[Q][Q], s_P[Q][Q];
  __shared__ float s_b[Q], s_g[Q], s_f[Q];      // beta, the decays and their products up to a token (one number for all channels)
  const int b = blockIdx.x, h = blockIdx.y, e = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int cnt = m.ent_count[e], start = m.ent_start[e], t0 = b * Q, left = cnt - t0;
  if (left <= 0) return;
  const int kh = h / (a.heads / a.kv_heads);
  const RecBlockLayout lay(a.dim, a.vdim, SOLVE);
  float* out = scratch + ((size_t)(rec_first_block(start, e) + b) * a.heads + h) * lay.stride;
  const size_t tok0 = (size_t)(start + t0);
  float x[Q];      // a column of the system: a value channel's numbers are on their way from here on
  auto values = [&](int ecol) {
    const float* vp = a.v + (size_t)h * a.vdim + min(ecol, a.vdim - 1);
#pragma unroll
    for (int t = 0; t < Q; t++) x[t] = vp[(tok0 + min(t, left - 1)) * a.ldv];
  };
  if (tid >= DP) values(tid - DP);
#pragma unroll
  for (int u = 0; u < Q * R4 / 256; u++) {
    const int i = tid + 256 * u, t = i / R4, d = 4 * (i % R4);
    const size_t tok = tok0 + min(t, left - 1);
    const bool in = t < left && d < a.dim;
    const int dc = min(d, a.dim - 4);
    const f32x4 qv = *reinterpret_cast<const f32x4*>(a.a + tok * a.lda + (size_t)kh * a.dim + dc), kv = *reinterpret_cast<const f32x4*>(a.k + tok * a.ldk + (size_t)kh * a.dim + dc);
    f32x4 wv4 = {1.f, 1.f, 1.f, 1.f};
    if constexpr (!SCALAR) wv4 = *reinterpret_cast<const f32x4*>(a.w + tok * a.ldw + (size_t)(KIND == REC_CDELTA ? h : kh) * a.dim + dc);
#pragma unroll
    for (int c = 0; c < 4; c++) {
      s_q[t][d + c] = in ? qv[c] : 0.f;
      s_k[t][d + c] = in ? kv[c] : 0.f;
      if constexpr (!SCALAR) s_w[t][d + c] = in ? wv4[c] : 1.f;
    }
  }
  for (int i = tid; i < Q * Q; i += 256) s_P[i / Q][i % Q] = 0.f;
  if (SOLVE && tid < Q) {
    const size_t at = (tok0 + min(tid, left - 1)) * a.ldg + h;
    s_b[tid] = tid < left ? a.beta[at] : 0.f;
    if constexpr (SCALAR) s_g[tid] = tid < left ? a.g[at] : 1.f;
  }
  __syncthreads();
  {
    const int dg = lane & 7, w8 = 8 * ((wv + b) & 3), i = w8 + (lane >> 3);      // (the wave with the earliest tokens has most pairs: not the same SIMD's in every block)
    auto row = [&](const float (*s)[DP], int t, f32x4* v) {      // this lane's channels 32 j + 4 dg + 0 .. 3: the eight lanes of a pair read one run of a row
#pragma unroll
      for (int j = 0; j < DPT / 4; j++) v[j] = *reinterpret_cast<const f32x4*>(&s[t][32 * j + 4 * dg]);
    };
    auto dot = [&](const f32x4* x, const f32x4* y) -> double {      // four sums side by side
      f32x4 s = x[0] * y[0];
#pragma unroll
      for (int j = 1; j < DPT / 4; j++)
#pragma unroll
        for (int c = 0; c < 4; c++) s[c] = fmaf(x[j][c], y[j][c], s[c]);
      return row_sum8(((double)s[0] + (double)s[1]) + ((double)s[2] + (double)s[3]));
    };
    f32x4 r[DPT / 4], qi[DPT / 4];
    row(s_k, i, r);
    row(s_q, i, qi);
    if constexpr (KIND == REC_WKV) {      // the token's own bonus
#pragma unroll
      for (int j = 0; j < DPT / 4; j++) {
        const int d = 32 * j + 4 * dg;
#pragma unroll
        for (int c = 0; c < 4; c++) qi[j][c] *= d + c < a.dim ? a.u[(size_t)h * a.dim + d + c] : 0.f;
      }
    }
    const float own = (float)dot(qi, r);
    if (dg == 0) s_P[i][i] = own;
    double c = 1.0;
    struct Rows { f32x4 q[DPT / 4], k[SOLVE ? DPT / 4 : 1], w[SCALAR ? 1 : DPT / 4]; };
    auto take = [&](Rows& o, int t) {
      row(s_q, t, o.q);
      if constexpr (SOLVE) row(s_k, t, o.k);
      if constexpr (!SCALAR) row(s_w, KIND == REC_WKV ? t - 1 : t, o.w);
    };
    auto pair = [&](const Rows& o, int t) {
      const bool on = t > i && (KIND != REC_WKV || t > i + 1);      // (wkv: the decays up to t - 1)
      if constexpr (SCALAR) c = t > i ? c * (double)s_g[t] : 1.0;
      else
#pragma unroll
        for (int j = 0; j < DPT / 4; j++)
#pragma unroll
          for (int x = 0; x < 4; x++) r[j][x] *= on ? o.w[j][x] : 1.f;
      const double p = dot(o.q, r);
      if constexpr (SOLVE) {
        const double k = dot(o.k, r);
        if (dg == 0 && t > i) s_A[i][t] = s_b[t] * (float)(SCALAR ? k * c : k);
      }
      if (dg == 0 && t > i) s_P[t][i] = (float)(SCALAR ? p * c : p);
    };
    Rows ra, rb;      // (wave-uniform bounds: a lane waits for its token; a token's rows are on their way one token ahead)
    take(ra, w8 + 1);
    for (int t = w8 + 1; t < Q; t += 2) {      // (an odd number of tokens)
      take(rb, min(t + 1, Q - 1));
      pair(ra, t);
      take(ra, min(t + 2, Q - 1));
      if (t + 1 < Q) pair(rb, t + 1);
    }
    if (SCALAR && tid < Q) {
      double f = 1.0;
      for (int t = 0; t <= tid; t++) f *= (double)s_g[t];
      s_f[tid] = (float)f;
    }
  }
  __syncthreads();
  // columns: the key channels (decayed rows, W), then the value channels (U)
  for (int col = tid; col < DP + lay.ep; col += 256) {
    const bool key = col < DP;
    const int ecol = col - DP;
    if (key) {
      const int d = col;
      double suf = 1.0;
      float* kd = out + lay.k + (size_t)(d >> 4) * 512 + (d & 15) * 4;
#pragma unroll
      for (int t4 = Q / 4 - 1; t4 >= 0; t4--) {
        f32x4 v;
#pragma unroll
        for (int u = 3; u >= 0; u--) { const int t = 4 * t4 + u; v[u] = s_k[t][d] * (float)suf; suf *= (double)(SCALAR ? s_g[t] : s_w[t][d]); }
        *reinterpret_cast<f32x4*>(kd + (t4 >> 2) * 256 + (t4 & 3) * 64) = v;
      }
      out[lay.g + d] = (float)suf;
      double f = 1.0;
#pragma unroll
      for (int t = 0; t < Q; t++) {
        if (KIND == REC_WKV) { const float wt = s_w[t][d]; s_w[t][d] = (float)f; f *= (double)wt; }      // (q takes the decays up to the token before)
        else {
          f *= (double)(SCALAR ? s_g[t] : s_w[t][d]);
          if constexpr (!SCALAR) s_w[t][d] = (float)f;
          x[t] = s_b[t] * (s_k[t][d] * (float)f);
        }
      }
    } else {
      if (col >= 256) values(ecol);
#pragma unroll
      for (int t = 0; t < Q; t++) x[t] = t < left && ecol < a.vdim ? (SOLVE ? s_b[t] * x[t] : x[t]) : 0.f;
    }
    if constexpr (SOLVE) {      // a known token goes to the equations of all later ones: no chain but from token to token; the next column of A is on its way
      float gone[Q];      // what the tokens before take from an equation
#pragma unroll
      for (int t = 0; t < Q; t++) gone[t] = 0.f;
      auto column = [&](f32x4* c, int i) {
#pragma unroll
        for (int q = (i + 1) / 4; q < Q / 4; q++) c[q] = *reinterpret_cast<const f32x4*>(&s_A[i][4 * q]);
      };
      f32x4 c0[Q / 4], c1[Q / 4];
      auto leave = [&](const f32x4* c, int i) {
        x[i] -= gone[i];
#pragma unroll
        for (int t = i + 1; t < Q; t++) gone[t] = fmaf(c[t / 4][t & 3], x[i], gone[t]);
      };
      column(c0, 0);
#pragma unroll
      for (int i = 0; i < Q; i += 2) {
        column(c1, i + 1);
        leave(c0, i);
        if (i + 2 < Q) column(c0, i + 2);
        leave(c1, i + 1);
        __builtin_amdgcn_sched_barrier(0);      // (two columns at a time in registers, not all)
      }
    }
    if (key) {
      if constexpr (SOLVE)
#pragma unroll
        for (int t = 0; t < Q; t++) s_k[t][col] = x[t];
    } else {
      float* ud = out + lay.u + (size_t)(ecol >> 4) * 512 + (ecol & 15) * 4;
#pragma unroll
      for (int t4 = 0; t4 < Q / 4; t4++) *reinterpret_cast<f32x4*>(ud + (t4 >> 2) * 256 + (t4 & 3) * 64) = f32x4{x[4 * t4], x[4 * t4 + 1], x[4 * t4 + 2], x[4 * t4 + 3]};
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < Q * R4 / 256; u++) {
    const int f = tid + 256 * u, ln = f & 63, tile = (f >> 6) & 1, dt = f >> 7, t = 16 * tile + (ln & 15), d = 16 * dt + 4 * (ln >> 4);
    f32x4 qv = *reinterpret_cast<const f32x4*>(&s_q[t][d]);
    if constexpr (SCALAR) qv *= s_f[t];
    else qv *= *reinterpret_cast<const f32x4*>(&s_w[t][d]);
    *reinterpret_cast<f32x4*>(out + lay.q + 4 * (size_t)f) = qv;
    if constexpr (SOLVE) *reinterpret_cast<f32x4*>(out + lay.w + 4 * (size_t)f) = *reinterpret_cast<const f32x4*>(&s_k[t][d]);
  }
  {
    const int rr = tid >> 6, t = tid & 15, g = (tid >> 4) & 3;      // [i % 4][lane][2 (t / 16) + i / 16]
    f32x4 v;
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = s_P[t + 16 * (k >> 1)][16 * (k & 1) + 4 * g + rr];
    *reinterpret_cast<f32x4*>(out + lay.p + 4 * (size_t)tid) = v;
  }
}

// NT: 16-channel tiles of the state per wave (64 NT key channels).  Wave w owns the state rows of its tiles and 16 columns, in the accumulator layout: register r of lane l is row
// 4 (l / 16) + r, column l % 16.  That is at the same time a B operand whose contraction slots are those rows, so W S and Q S need no transposition, and the same holds for u, whose
// rows are tokens.  The four waves' shares of W S (and, a block later, of the outputs) meet in LDS; two buffers each, one barrier a block.  A block's operands are asked for a block
// ahead, straight into registers: no wave reads another's.  Grid: (entries, heads, E / 16).
// DEPTH: blocks whose operands are in registers or on their way.  Two, so that a compute unit has room for two workgroups; three for wkv heads of more than 64 channels, whose block has
// the fewest matrix instructions for its bytes.  2048 tokens, two / three, us: wkv 64 x 64 48 / 54, 128 x 128 85 / 72, delta rules 128 x 128 109 / 112, eight entries of 300 tokens and 16
// heads 60 / 84.
template <int KIND, int NT>
constexpr int rec_block_depth() { return KIND == REC_WKV && NT == 2 ? 3 : 2; }
template <int KIND, int NT, int DEPTH = rec_block_depth<KIND, NT>()>
__global__ __launch_bounds__(256, DEPTH > 2 ? 1 : 2) void rec_block_kernel(StepMeta m, RecScanArgs a, const float* scratch) {
  constexpr int Q = REC_BLOCK;
  constexpr bool SOLVE = KIND != REC_WKV;
  __shared__ __attribute__((aligned(16))) f32x4 s_u[2][4][2][64], s_o[2][4][2][64];
  const int e = blockIdx.x, h = blockIdx.y, ct = blockIdx.z, tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), g4 = lane >> 4, l16 = lane & 15;
  const int cnt = m.ent_count[e], start = m.ent_start[e], slot = m.ent_row[e], nblk = (cnt + Q - 1) / Q;
  const bool fresh = m.tok_pos[start] == 0;
  const RecBlockLayout lay(a.dim, a.vdim, SOLVE);
  const float* base = scratch + ((size_t)rec_first_block(start, e) * a.heads + h) * lay.stride;
  const size_t bstride = (size_t)a.heads * lay.stride;
  const int j = ct * 16 + l16, wl = tid >> 6;      // (wl: the wave's number in a vector register, for selects instead of branches)
  const bool col = j < a.vdim;
  float* Sg = a.S + ((size_t)slot * a.heads + h) * (size_t)a.dim * a.vdim;
  f32x4 S[NT];
#pragma unroll
  for (int n = 0; n < NT; n++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int d = 16 * (wv * NT + n) + 4 * g4 + r;
      S[n][r] = !fresh && col && d < a.dim ? Sg[(size_t)d * a.vdim + j] : 0.f;
    }
  struct Ops { f32x4 q[NT][2], k[NT][2], w[SOLVE ? NT : 1][2], u[2], p, g[NT]; };
  auto four = [](const float* p, unsigned int floats) { return *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(p) + 4u * floats); };      // (one address for the wave, a lane's offset beside it)
  const unsigned int own = (unsigned int)(wv * NT * 512 + 4 * lane);
  auto fetch = [&](Ops& o, int b) {
    const float* s = base + (size_t)b * bstride;
    const float *sw = s + lay.w, *sq = s + lay.q, *sk = s + lay.k;
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
      for (int t = 0; t < 2; t++) {
        if constexpr (SOLVE) o.w[n][t] = four(sw, own + 512u * n + 256u * t);
        o.q[n][t] = four(sq, own + 512u * n + 256u * t);
      }
#pragma unroll
    for (int t = 0; t < 2; t++) o.u[t] = four(s + lay.u, 512u * ct + 256u * t + 4u * lane);
#pragma unroll
    for (int n = 0; n < NT; n++) {
      o.g[n] = four(s + lay.g, 16u * (wv * NT + n) + 4u * g4);
#pragma unroll
      for (int t = 0; t < 2; t++) o.k[n][t] = four(sk, own + 512u * n + 256u * t);
    }
    o.p = four(s + lay.p, 256u * wv + 4u * lane);
  };
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto lds_barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); __builtin_amdgcn_s_barrier(); };      // (loads of the blocks ahead and stores stay on their way)
  // outputs of block b: wave w takes rows 4 g + 2 (w % 2) + 0, 1 of token tile w / 2
  const int tok_l = 16 * (wl >> 1) + 4 * g4 + 2 * (wl & 1);
  const unsigned int out_l = (unsigned int)tok_l * (unsigned int)a.ldo + (unsigned int)l16;
  float* outb = a.out + (size_t)start * a.ldo + (size_t)h * a.vdim + ct * 16;
  auto store = [&](int b) {
    const f32x2 *p = reinterpret_cast<const f32x2*>(&s_o[b & 1][0][wv >> 1][lane]) + (wv & 1);
    const f32x2 v = (p[0] + p[256]) + (p[512] + p[768]);
    char* o = reinterpret_cast<char*>(outb + (size_t)max(b, 0) * Q * a.ldo);
    const int tok = b * Q + tok_l;
    if (b >= 0 && col) {
      if (tok < cnt) *reinterpret_cast<float*>(o + 4u * out_l) = v[0];
      if (tok + 1 < cnt) *reinterpret_cast<float*>(o + 4u * (out_l + (unsigned int)a.ldo)) = v[1];
    }
  };
  auto block = [&](const Ops& o, int b) {
    f32x4 acc[2][NT];
    if constexpr (SOLVE) {
      f32x4 us[2][NT];
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int n = 0; n < NT; n++) us[t][n] = zero;
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
          for (int t = 0; t < 2; t++) us[t][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[n][t][r], S[n][r], us[t][n], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 2; t++) {
        f32x4 v = us[t][0];
#pragma unroll
        for (int n = 1; n < NT; n++) v += us[t][n];
        s_u[b & 1][wv][t][lane] = v;
      }
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int n = 0; n < NT; n++) acc[t][n] = zero;
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int t = 0; t < 2; t++) acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[n][t][r], S[n][r], acc[t][n], 0, 0, 0);
    lds_barrier();      // the shares of this block's W S stand, and the outputs' of the block before
    f32x4 u[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      u[t] = o.u[t];
      if constexpr (SOLVE) u[t] -= (s_u[b & 1][0][t][lane] + s_u[b & 1][1][t][lane]) + (s_u[b & 1][2][t][lane] + s_u[b & 1][3][t][lane]);
    }
#pragma unroll
    for (int n = 0; n < NT; n++) S[n] *= o.g[n];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int n = 0; n < NT; n++) S[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.k[n][t][r], u[t][r], S[n], 0, 0, 0);
    // the block's own tokens: this wave's are those with i % 4 = its number
    const float u0 = wl & 2 ? (wl & 1 ? u[0][3] : u[0][2]) : (wl & 1 ? u[0][1] : u[0][0]), u1 = wl & 2 ? (wl & 1 ? u[1][3] : u[1][2]) : (wl & 1 ? u[1][1] : u[1][0]);
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
      for (int n = 1; n < NT; n++) acc[t][0] += acc[t][n];
      acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.p[2 * t], u0, acc[t][0], 0, 0, 0);
      if (t > 0) acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.p[2 * t + 1], u1, acc[t][0], 0, 0, 0);      // (the second half's tokens are ahead of the first's)
      s_o[b & 1][wv][t][lane] = acc[t][0];
    }
    store(b - 1);      // (block 0 has none before it)
  };
  Ops o[DEPTH];
#pragma unroll
  for (int k = 0; k + 1 < DEPTH; k++) { fetch(o[k], min(k, nblk - 1)); __builtin_amdgcn_sched_barrier(0); }      // (in order: a block waits for its own loads only)
  auto turn = [&](auto Kc, int b) {
    constexpr int k = decltype(Kc)::value;
    fetch(o[(k + DEPTH - 1) % DEPTH], min(b + DEPTH - 1, nblk - 1));      // (past the end: the last one again, not used)
    __builtin_amdgcn_sched_barrier(0);
    block(o[k], b);
    __builtin_amdgcn_sched_barrier(0);
  };
  using std::integral_constant;
  int b = 0;
  for (; b + DEPTH <= nblk; b += DEPTH) {
    turn(integral_constant<int, 0>{}, b);
    turn(integral_constant<int, 1>{}, b + 1);
    if constexpr (DEPTH > 2) turn(integral_constant<int, 2>{}, b + 2);
  }
  if (b < nblk) block(o[0], b++);
  if (DEPTH > 2 && b < nblk) block(o[1], b);
  lds_barrier();
  store(nblk - 1);
#pragma unroll
  for (int n = 0; n < NT; n++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int d = 16 * (wv * NT + n) + 4 * g4 + r;
      if (col && d < a.dim) Sg[(size_t)d * a.vdim + j] = S[n][r];
    }
}

}  // namespace tgx
