// stack_rec.h — row-wise kernels of the layered designs whose layers run a mixer and a feed-forward side by side behind ONE norm, and whose mixers keep
// a decaying matrix state per head (Vitudra).  Same conventions as stack.h / stack_seq.h: a step's T tokens are the concatenated entries of a ragged
// batch (StepMeta), all arithmetic here is fp32, every reduction has a fixed order.
//   offset_norm_kernel      rows / sqrt(mean(row^2) + eps) * (offset + w): an RMS norm whose weight is stored as its distance from `offset`
//   token_shift_kernel      the n mixes h + (h_before - h) * mu_s of a token-shift layer, and the slot's last row
//   delta_prep_kernel       causal depth-wise convolution + silu on the q | k | v projections of a gated-delta-rule layer (tails per slot), unit q and k per
//                           head, beta = sigmoid, decay = exp(-exp(A_log) * softplus(a + dt_bias)) (where the layer has one decay per head)
//   rec_scan_kernel         the recurrence over an entry's tokens with the head's matrix state in registers:
//                             REC_WKV     o = (S + diag(u) k v^T)^T r;  S <- diag(w) S + k v^T
//                             REC_DELTA   S <- g S;  S += k (beta (v - S^T k))^T;  o = S^T q
//                             REC_SSD     S <- g S + k (beta v)^T;  o = S^T q + skip v (a scalar-decay state-space recurrence; with `fixed`, a retention:
//                                         the decay is a number per head and beta one number)
//                             REC_CDELTA  S <- diag(w) S;  S += k (beta (v - S^T k))^T;  o = S^T q (the delta rule with one decay per head and key channel)
// A sequence whose first token has position 0 starts from zero state whatever its slot held.
#pragma once
#include "stack.h"
#include "stack_rec_args.h"

namespace tgx {

// out[i] = x[rows ? rows[i] : i] / sqrt(mean(row^2) + eps) * (offset + w)
__global__ __launch_bounds__(256) void offset_norm_kernel(const float* x, const int* rows, const float* w, float offset, float* out, int W, float eps, RowTerms terms) {
  __shared__ float s4[4];
  const float* xr = x + (size_t)(rows ? rows[blockIdx.x] : blockIdx.x) * W;
  float* o = out + (size_t)blockIdx.x * W;
  float ss = 0.f;
  if ((W & 3) == 0 && W <= 1024 * ROW_REG) {      // (the weights are on their way before the sum)
    f32x4 v[ROW_REG], wv[ROW_REG];
#pragma unroll
    for (int k = 0; k < ROW_REG; k++) { v[k] = row_load<true>(xr, k, W); wv[k] = row_load<true>(w, k, W); }
#pragma unroll
    for (int k = 0; k < ROW_REG; k++)
#pragma unroll
      for (int u = 0; u < 4; u++) ss = fmaf(v[k][u], v[k][u], ss);
    const float r = 1.0f / sqrtf(block_sum_once(ss, s4) / (float)W + eps);
#pragma unroll
    for (int k = 0; k < ROW_REG; k++) {
      for (int u = 0; u < 4; u++) v[k][u] = v[k][u] * r * (offset + wv[k][u]);
      row_store<true>(o, k, W, v[k]);
      if (terms.out) row_store_terms(terms, blockIdx.x, k, W, v[k]);
    }
    return;
  }
  for (int c = threadIdx.x; c < W; c += 256) ss = fmaf(xr[c], xr[c], ss);
  ss = block_sum_256(ss, s4);
  const float r = 1.0f / sqrtf(ss / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += 256) o[c] = xr[c] * r * (offset + w[c]);
}

// ---- token shift.  One thread per (token, channel): out[t][s] = h_t + (h_(t-1) - h_t) * mu[s] for the n mixes; h_(t-1) is the row before in the entry,
// the slot's kept row for an entry's first token, zero at position 0.  The kept row is double-buffered with the slot's step parity (the entry's last
// token writes buffer par ^ 1 while its first reads buffer par).  Grid: (tokens, width / 256).
// NORM: h is the stream in front of the layer's RMS norm (eps, offset + w), which every workgroup makes for itself: one launch where the norm and the shift were two (a decoded row of
// 1024 channels: 2.3 + 2.9 us, here 3.2; 3.7 with a channel, then a mix, after the other).
struct TokenShiftArgs {
  const float* h;        // [T][W]
  const float* mu;       // [n][W]
  float* out;            // [T][n][W]
  float* state;          // [2][slots][W]
  size_t state_buf;
  int W, n;
  const float* w; float offset, eps;
};
template <bool NORM>
__global__ __launch_bounds__(256) void token_shift_kernel(StepMeta m, TokenShiftArgs a) {
  constexpr int MU = 8, RV = 8;      // mixes, and channels a thread of a row's sum, that are on their way at once, the row's and the mixes' in front of what the tables say
  __shared__ float s_now[4], s_before[4];
  const int t = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (!NORM && c >= a.W) return;
  const int cc = min(c, a.W - 1);
  const float* __restrict__ cur = a.h + (size_t)t * a.W;
  const float* __restrict__ mus = a.mu + cc;
  float* __restrict__ outp = a.out + (size_t)t * a.n * a.W;
  float mu[MU];
#pragma unroll
  for (int s = 0; s < MU; s++) mu[s] = mus[(size_t)min(s, a.n - 1) * a.W];
  float x = cur[cc];
  const float w = NORM ? a.offset + a.w[cc] : 1.f;
  auto squares = [&](const float* __restrict__ r, int k0) {
    float v[RV], ss = 0.f;
#pragma unroll
    for (int k = 0; k < RV; k++) v[k] = r[min(k0 + 256 * k, a.W - 1)];
#pragma unroll
    for (int k = 0; k < RV; k++) if (k0 + 256 * k < a.W) ss = fmaf(v[k], v[k], ss);
    return ss;
  };
  const int i = m.tok_idx[t], cnt = m.tok_cnt[t], pos = m.tok_pos[t], row = m.tok_row[t], par = m.tok_par[t];
  const float* __restrict__ before = i > 0 ? cur - a.W : a.state + (size_t)par * a.state_buf + (size_t)row * a.W;
  float b = pos == 0 ? 0.f : before[cc];
  if constexpr (NORM) {
    auto factor = [&](const float* r, float* s4) {
      float ss = 0.f;
      for (int k0 = threadIdx.x; k0 < a.W; k0 += 256 * RV) ss += squares(r, k0);
      return 1.0f / sqrtf(block_sum_once(ss, s4) / (float)a.W + a.eps);
    };
    x = x * factor(cur, s_now) * w;
    if (i > 0) b = b * factor(before, s_before) * w;      // (a row of this step: its own norm; the slot's is normed)
    if (c >= a.W) return;
  }
  const float d = b - x;
  for (int s0 = 0; s0 < a.n; s0 += MU) {
    if (s0 > 0)
#pragma unroll
      for (int s = 0; s < MU; s++) mu[s] = mus[(size_t)min(s0 + s, a.n - 1) * a.W];
#pragma unroll
    for (int s = 0; s < MU; s++) if (s0 + s < a.n) outp[(size_t)(s0 + s) * a.W + c] = fmaf(d, mu[s], x);
  }
  if (i == cnt - 1) a.state[(size_t)(par ^ 1) * a.state_buf + (size_t)row * a.W + c] = x;
}

// ---- inputs of a gated-delta-rule layer.  proj row = [.. | q (G D) | k (G D) | v (H E) | b (H) | a (H) | ..] from column col0; the C = 2 G D + H E
// convolved channels take taps weights each (last = the current token's); the taps - 1 rows before come from the step's own rows, the slot's tails (raw
// projections, double-buffered by step parity like the other per-slot rows) or are zero before the sequence's start.
// out row = [q | k | v | beta | decay]: q, k unit vectors per head (x / sqrt(sum x^2 + unit_eps)), q times q_scale.  The b columns stand at b_col (from col0); a layer
// without a_log has no scalar decays (neither a columns nor decay outputs).
// Grid: (tokens, 2 G + H + 1): one workgroup per q head, k head (D <= 256 channels, one per thread, and their norm), v head, and one for the H gates.
constexpr int DELTA_MAX_TAPS = 64;      // (bounds the per-slot tails, not the kernel: it loops over the taps)
struct DeltaPrepArgs {
  const float* proj; long long ldp; int col0, b_col;
  const float* cw;       // [C][taps]
  const float* a_log;    // [H] (nullptr: no scalar decays)
  const float* dt_bias;  // [H]
  float* out; long long ldo;
  float* state;          // [2][slots][taps - 1][C] (nullptr when taps == 1)
  size_t state_buf;
  int heads, kv_heads, dim, vdim, taps;
  float q_scale, unit_eps;
};
__global__ __launch_bounds__(256) void delta_prep_kernel(StepMeta m, DeltaPrepArgs a) {
  __shared__ float s4[4];
  const int t = blockIdx.x, u = blockIdx.y, i = m.tok_idx[t], cnt = m.tok_cnt[t], pos = m.tok_pos[t], row = m.tok_row[t], par = m.tok_par[t];
  const int G2 = 2 * a.kv_heads, GD = a.kv_heads * a.dim, C = 2 * GD + a.heads * a.vdim, nb = a.taps - 1;
  const float* __restrict__ pr = a.proj + (size_t)t * a.ldp + a.col0;
  float* __restrict__ o = a.out + (size_t)t * a.ldo;
  if (u == G2 + a.heads) {
    for (int h = threadIdx.x; h < a.heads; h += 256) {
      o[C + h] = 1.0f / (1.0f + expf(-pr[a.b_col + h]));
      if (!a.a_log) continue;
      const float za = pr[a.b_col + a.heads + h] + a.dt_bias[h];
      const float sp = za > 20.f ? za : log1pf(expf(za));
      o[C + a.heads + h] = expf(-expf(a.a_log[h]) * sp);
    }
    return;
  }
  const bool qk = u < G2;
  const int n = qk ? a.dim : a.vdim, c0 = qk ? u * a.dim : 2 * GD + (u - G2) * a.vdim;
  const float* __restrict__ st_old = a.state ? a.state + (size_t)par * a.state_buf + (size_t)row * nb * C : nullptr;
  float* __restrict__ st_new = a.state ? a.state + (size_t)(par ^ 1) * a.state_buf + (size_t)row * nb * C : nullptr;
  const float* __restrict__ cw = a.cw;
  float mine = 0.f;                                        // a q / k head's channel of this thread (D <= 256)
  for (int cc = threadIdx.x; cc < n; cc += 256) {
    const int c = c0 + cc;
    const float x0 = pr[c];
    float acc = cw[(size_t)c * a.taps + nb] * x0;
    for (int d = 1; d <= nb; d++) {                        // the row d positions back
      float xv = 0.f;
      if (d <= i) xv = pr[c - (long long)d * a.ldp];
      else if (pos - d >= 0) xv = st_old[(size_t)(nb - (d - i)) * C + c];      // tail slot s holds position past - nb + s, past = pos - i
      acc = fmaf(cw[(size_t)c * a.taps + nb - d], xv, acc);
    }
    const float act = acc / (1.0f + expf(-acc));
    if (qk) mine = act; else o[c] = act;
    if (st_new) {
      const int s = nb - (cnt - i);                        // row i of cnt lands in tail slot nb - (cnt - i) ...
      if (s >= 0) st_new[(size_t)s * C + c] = x0;
      if (i == 0)                                          // ... and an entry shorter than the tails keeps the end of the old ones
        for (int k = 0; k + cnt < nb; k++) st_new[(size_t)k * C + c] = (pos - (nb - cnt - k) >= 0) ? st_old[(size_t)(k + cnt) * C + c] : 0.f;
    }
  }
  if (!qk) return;
  const float ss = block_sum_256(mine * mine, s4);
  const float r = (u < a.kv_heads ? a.q_scale : 1.0f) / sqrtf(ss + a.unit_eps);
  if ((int)threadIdx.x < n) o[c0 + threadIdx.x] = mine * r;
}

// ---- the recurrences.  One workgroup per (entry, head, 256 / RG value columns) walks the entry's tokens in order, TB at a time: the block's per-key-channel
// inputs (up to three vectors of `dim`) and the workgroup's value columns are staged in LDS (the next block's travel in registers meanwhile), then every
// lane updates its DPER rows of its column with no barrier inside the block: a wave's lanes = 64 / RG columns x RG row groups (the row groups of a column are
// adjacent lanes), RG DPER >= dim.  Sums over the key channels cross the row groups on the lane crossbar.
// What bounds a prompt is the instructions that one wave issues per token, four cycles each, and the waits between dependent ones where a SIMD has a single wave.  So a step that
// leaves compute units idle spreads a column over more row groups (sixteen, or thirty-two of four rows: twice the workgroups of half the rows), a full chip takes eight, which issue
// fewer instructions in all; two tokens go without a branch between them, so that the one's sum over the groups lies under the other's arithmetic; and a column's outputs are kept by its
// row groups, a token each, and leave in one store for as many tokens as there are groups.  2048 tokens, delta rule of 16 heads of 128 x 128: 632 us at eight row groups staged number
// by number, 578 staged in vectors of four, 470 at sixteen with a store a token, 340 at thirty-two and stores by the block; wkv of 32 heads of 64 x 64 419, 409, 335, 257 (sixteen groups).
constexpr int rec_cols(int rg) { return 4 * (64 / rg); }      // columns per workgroup
template <int DPER, int KIND, int RG, bool VEC>
__global__ __launch_bounds__(256) void rec_scan_kernel(StepMeta m, RecScanArgs a) {
  constexpr int CW = 64 / RG, CB = rec_cols(RG), LP = RG >= 16 && DPER == 4 ? 4 : DPER + 4, DP = RG * DPER, TB = DP <= 128 ? 16 : 8;      // LP: a row group's LDS stride (the groups' reads fall into different banks)
  constexpr int Q4 = TB * DP / 4, NQ = (Q4 + 255) / 256, NV = (TB * CB + 255) / 256, NA = KIND == REC_WKV || KIND == REC_CDELTA ? 3 : 2;
  __shared__ __attribute__((aligned(16))) float s_in[NA][TB][RG * LP];      // [0]: the read vector, [1]: k, [2]: the decay
  __shared__ float s_v[TB][CB], s_b[TB], s_g[TB];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, rg = lane % RG, cl = lane / RG;
  const int jl = wv * CW + cl, j = blockIdx.z * CB + jl;
  const int start = m.ent_start[e], cnt = m.ent_count[e], row = m.ent_row[e];
  const bool fresh = m.tok_pos[start] == 0;
  const int kh = h / (a.heads / a.kv_heads), d0 = rg * DPER, l0 = rg * LP;
  const bool col = j < a.vdim;
  float* Sg = a.S + ((size_t)row * a.heads + h) * (size_t)a.dim * a.vdim;
  const float skip = KIND == REC_SSD && a.skip ? a.skip[h] : 0.f;
  float S[DPER], ub[KIND == REC_WKV ? DPER : 1];
#pragma unroll
  for (int dd = 0; dd < DPER; dd++) {
    const int d = d0 + dd;
    S[dd] = (!fresh && d < a.dim && col) ? Sg[(size_t)d * a.vdim + j] : 0.f;
    if (KIND == REC_WKV) ub[dd] = d < a.dim ? a.u[(size_t)h * a.dim + d] : 0.f;
  }
  const float* src[3] = {a.a, a.k, a.w};
  const long long lds[3] = {a.lda, a.ldk, a.ldw};
  f32x4 rin[NA][NQ];
  float rv[NV], rb = 0.f, rgt = 0.f;
  auto fetch = [&](int t0) {
    const int nb = min(TB, cnt - t0);
#pragma unroll
    for (int u = 0; u < NQ; u++) {      // (rows past the entry's end repeat its last one and are never used)
      const int i = tid + 256 * u, t = min(i / (DP / 4), TB - 1), d = 4 * (i % (DP / 4));
      const size_t tok = (size_t)(start + min(t0 + t, cnt - 1));
#pragma unroll
      for (int s = 0; s < NA; s++) {
        const float* p = src[s] + tok * lds[s] + (size_t)(KIND == REC_CDELTA && s == 2 ? h : kh) * a.dim;
        if constexpr (VEC) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(p + min(d, a.dim - 4));
#pragma unroll
          for (int c = 0; c < 4; c++) rin[s][u][c] = d < a.dim ? v[c] : 0.f;
        } else
#pragma unroll
          for (int c = 0; c < 4; c++) { const float v = p[min(d + c, a.dim - 1)]; rin[s][u][c] = d + c < a.dim ? v : 0.f; }
      }
    }
#pragma unroll
    for (int u = 0; u < NV; u++) {
      const int i = tid + 256 * u, t = i / CB, c = i - t * CB;
      rv[u] = (t < nb && blockIdx.z * CB + c < a.vdim) ? a.v[(size_t)(start + t0 + t) * a.ldv + (size_t)h * a.vdim + blockIdx.z * CB + c] : 0.f;
    }
    if (KIND != REC_WKV && tid < nb) {
      const size_t at = (size_t)(start + t0 + tid) * a.ldg + h;
      if (KIND == REC_SSD && a.fixed) { rb = a.beta0; rgt = a.fixed[h]; }
      else { rb = a.beta[at]; if (KIND != REC_CDELTA) rgt = a.g[at]; }
    }
  };
  fetch(0);
  for (int t0 = 0; t0 < cnt; t0 += TB) {
    const int nb = min(TB, cnt - t0);
    __syncthreads();                                       // the block before has been read
#pragma unroll
    for (int u = 0; u < NQ; u++) {
      const int i = tid + 256 * u, t = i / (DP / 4), d = 4 * (i - t * (DP / 4)), at = (d / DPER) * LP + d % DPER;
#pragma unroll
      for (int s = 0; s < NA; s++) if (i < Q4) *reinterpret_cast<f32x4*>(&s_in[s][t][at]) = rin[s][u];
    }
#pragma unroll
    for (int u = 0; u < NV; u++) { const int i = tid + 256 * u; if (i < TB * CB) s_v[i / CB][i % CB] = rv[u]; }
    if (KIND != REC_WKV && tid < TB) { s_b[tid] = rb; s_g[tid] = rgt; }
    __syncthreads();
    if (t0 + TB < cnt) fetch(t0 + TB);
    // a token's operands travel from LDS to registers one token ahead of their use (two register sets, taken in turn), so the reads' latency lies under
    // the arithmetic of the token before instead of on the recurrence's critical path
    struct Tok { f32x4 in[NA][DPER / 4]; float v, g, b; };
    auto take = [&](Tok& k, int t) {
#pragma unroll
      for (int s = 0; s < NA; s++)
#pragma unroll
        for (int dd = 0; dd < DPER; dd += 4) k.in[s][dd / 4] = *reinterpret_cast<const f32x4*>(&s_in[s][t][l0 + dd]);
      k.v = s_v[t][jl];
      if (KIND != REC_WKV) { k.g = s_g[t]; k.b = s_b[t]; }
    };
    auto advance = [&](const Tok& k) -> float {
      float po = 0.f;
      if (KIND == REC_WKV) {
#pragma unroll
        for (int dd = 0; dd < DPER; dd++) {
          const float kv = k.in[1][dd / 4][dd & 3] * k.v;
          po = fmaf(k.in[0][dd / 4][dd & 3], fmaf(ub[dd], kv, S[dd]), po);
          S[dd] = fmaf(k.in[NA - 1][dd / 4][dd & 3], S[dd], kv);
        }
      } else if (KIND == REC_SSD) {
        const float bv = k.b * k.v;
#pragma unroll
        for (int dd = 0; dd < DPER; dd++) { S[dd] = fmaf(k.g, S[dd], k.in[1][dd / 4][dd & 3] * bv); po = fmaf(S[dd], k.in[0][dd / 4][dd & 3], po); }
      } else {
        float pk = 0.f;
#pragma unroll
        for (int dd = 0; dd < DPER; dd++) { S[dd] *= KIND == REC_CDELTA ? k.in[NA - 1][dd / 4][dd & 3] : k.g; pk = fmaf(S[dd], k.in[1][dd / 4][dd & 3], pk); }
        pk = row_group_sum<RG>(pk);
        const float uj = k.b * (k.v - pk);
#pragma unroll
        for (int dd = 0; dd < DPER; dd++) { S[dd] = fmaf(k.in[1][dd / 4][dd & 3], uj, S[dd]); po = fmaf(S[dd], k.in[0][dd / 4][dd & 3], po); }
      }
      po = row_group_sum<RG>(po);
      if (KIND == REC_SSD) po = fmaf(skip, k.v, po);
      return po;
    };
    // Every row group of a column ends with a token's output: group r keeps that of token r (of as many tokens as there are groups), so a column's tokens leave in one store.
    // Two tokens a turn without a branch between them: the one's sum over the groups lies under the other's arithmetic.
    constexpr int FL = RG < TB ? RG : TB;
    Tok ka, kb;
    take(ka, 0);
    for (int s0 = 0; s0 < nb; s0 += FL) {
      const int n = min(FL, nb - s0);
      float keep = 0.f;
      int t = 0;
      for (; t + 1 < n; t += 2) {
        take(kb, s0 + t + 1);
        const float o0 = advance(ka);
        take(ka, min(s0 + t + 2, TB - 1));
        const float o1 = advance(kb);
        keep = rg == t ? o0 : rg == t + 1 ? o1 : keep;
      }
      if (t < n) {
        const float o0 = advance(ka);
        take(ka, min(s0 + t + 1, TB - 1));
        keep = rg == t ? o0 : keep;
      }
      if (rg < n && col) a.out[(size_t)(start + t0 + s0 + rg) * a.ldo + (size_t)h * a.vdim + j] = keep;
    }
  }
#pragma unroll
  for (int dd = 0; dd < DPER; dd++) { const int d = d0 + dd; if (d < a.dim && col) Sg[(size_t)d * a.vdim + j] = S[dd]; }
}

}  // namespace tgx
