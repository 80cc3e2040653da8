// stack_ssd_mfma.h — the scalar-decay state-space recurrence S_t = g_t S_(t-1) + B_t (dt_t x_t)^T, y_t = S_t^T C_t + D x_t over long portions, 64 tokens at a time on
// the fp32 matrix cores (v_mfma_f32_32x32x2_f32: nothing is rounded below fp32).
// With cs_i = log g_1 + .. + log g_i inside a block of 64 tokens, the recurrence unrolls to three products per block:
//   y_i = sum_{j <= i} (C_i . B_j) exp(cs_i - cs_j) dt_j x_j  +  exp(cs_i) S_in^T C_i  +  D x_i,      S_out = exp(cs_64) S_in + sum_j B_j (exp(cs_64 - cs_j) dt_j x_j)^T
//   ssd_gram_kernel     C_i . B_j of every block and group (all heads of a group share it)
//   ssd_block_kernel    one workgroup per (entry, head, 32 value channels) walks the entry's blocks with the state in matrix-core accumulators
//   gate_scan_kernel    a matrix memory's gates as the decays and factors of that recurrence
// The sums cs are kept in double: a difference of two sums must be as exact as a sum of few logarithms.  Blocks are counted from the entry's first token, and a block
// past the entry's end is padded by tokens with dt = 0 and log g = 0, which change nothing.
#pragma once
#include "prefill.h"
#include "stack_meta.h"

namespace tgx {

constexpr int SSD_BLOCK = 64;
struct SsdArgs {
  const float* row; long long ld;      // per token x (heads E), B and C (groups N each) from columns x0, b0 and c0
  int x0, b0, c0;                      // b0 and c0 multiples of 4
  const float* gates; long long ldgate;      // per token and head: dt from column dt_col, the logarithm of the decay from column log_col
  int dt_col, log_col;
  int heads, groups, N, E;             // N a multiple of 4
  float* gram;                         // [blocks][groups][64][64]
  const float* fixed; float dt0;       // [2][heads] decays and their logarithms that hold for every token, with dt0 as every token's dt (nullptr: per token, from gates)
  const float* skip;                   // [heads] (nullptr: none)
  float* S;                            // [slots][heads][N][E]
  float* out; long long ldo;           // [T][heads E]
  float* norm_S; size_t norm_buf;      // a second state N_t = g_t N_(t-1) + dt_t B_t, the sum that a matrix memory divides by: [2][slots][heads][N], norm_buf between the two (nullptr: none)
  float* norm_out; long long ldn;      // N_t . C_t: [T][heads]
  int portion, portions;               // blocks of a portion (portions > 1: the longest entry's; an entry may have fewer)
  int ranked;                          // SSD_WHOLE: entries longest first
  float* states;                       // [entries][portions][heads][tiles][ssd_state_elems]: what the portions before leave (SSD_STATES)
};
// the first block of an entry in `gram`: entries never share a block
__device__ __forceinline__ int ssd_first_block(int start, int e) { return start / SSD_BLOCK + e; }

// G[i][j] = C_i . B_j, one 32 x 32 tile per wave (the tile above the diagonal is never read).  A lane holds one row of either operand: four consecutive channels per
// load, channel 8 q + 4 (lane / 32) + u as the two contraction slots of step 4 q + u.  Eight sums run side by side and meet in pairs, as the scan's eight row groups do: one sum
// over all channels was most of a block's error (a matrix memory of 128 / 256 channels, against 64 bits: 1.9 / 2.2 times the scan's error with one sum, 1.0 with eight).
// Grid: (blocks of the longest entry, groups, entries).
template <int Q = SSD_BLOCK>
__global__ __launch_bounds__(256) void ssd_gram_kernel(StepMeta m, SsdArgs a) {
  const int b = blockIdx.x, g = blockIdx.y, e = blockIdx.z, cnt = m.ent_count[e], start = m.ent_start[e];
  static_assert(Q == 64, "four tiles of 32 x 32");
  if (b * Q >= cnt) return;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, half = lane >> 5, l31 = lane & 31, it = wv >> 1, jt = wv & 1;
  if (jt > it) return;
  const int i = b * Q + 32 * it + l31, j = b * Q + 32 * jt + l31;
  const float* cr = a.row + (size_t)(start + min(i, cnt - 1)) * a.ld + a.c0 + (size_t)g * a.N;
  const float* br = a.row + (size_t)(start + min(j, cnt - 1)) * a.ld + a.b0 + (size_t)g * a.N;
  f32x16 acc[8];
#pragma unroll
  for (int k = 0; k < 8; k++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[k][r] = 0.f;
  for (int q0 = 0; q0 < (a.N + 7) / 8; q0 += 2)
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int n = 8 * (q0 + k) + 4 * half;
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      const f32x4 cv = n < a.N ? *reinterpret_cast<const f32x4*>(cr + n) : z, bv = n < a.N ? *reinterpret_cast<const f32x4*>(br + n) : z;
#pragma unroll
      for (int u = 0; u < 4; u++) acc[4 * k + u] = __builtin_amdgcn_mfma_f32_32x32x2f32(cv[u], bv[u], acc[4 * k + u], 0, 0, 0);
    }
#pragma unroll
  for (int k = 4; k > 0; k /= 2)
#pragma unroll
    for (int j2 = 0; j2 < k; j2++) acc[j2] += acc[j2 + k];
  float* G = a.gram + ((size_t)(ssd_first_block(start, e) + b) * a.groups + g) * (Q * Q);
#pragma unroll
  for (int r = 0; r < 16; r++) G[(32 * it + (r & 3) + 8 * (r >> 2) + 4 * half) * Q + 32 * jt + l31] = acc[0][r];
}

// NW: 32-row tiles of the state per wave (4 NW 32 >= N).  Wave w owns the state rows n of its tiles and 32 columns, in the accumulator layout: register r of a lane is
// row (r & 3) + 8 (r >> 2) + 4 (lane / 32), column lane % 32.  Register r of the two half-waves is at the same time a B operand whose two contraction slots are those
// two rows, so S^T C needs no transposition: its A operand takes C's channels in that order.  A wave contributes its rows' share of S^T C and the share of sixteen
// keys j of the block's own product; the four waves' shares are added up in LDS.  Grid: (heads, E / 32, portions entries).
// Operands travel straight from memory to registers (every wave reads its own state rows only): B of a block is asked for at the block's start and used at its end,
// C and the Gram rows of the next block replace the present ones as soon as these are used up, so nothing is held twice.  Rows past the
// entry's end are clamped to its last one (what is read there twice meets dt = 0 or is not stored).
// NORM: the grid's last tile carries the second state: the recurrence with x = 1 in one column.
// Entries and heads that leave the chip idle: a chain of blocks, 6.6 us each on 72 workgroups (2048 tokens, 8 heads of 128 x 256).  So an entry's blocks are cut into portions, which two
// launches take at once: SSD_STATES the state that every portion but the last adds to a state of zero (the first: leaves behind the entry's own), and how much it decays; SSD_PORTIONS
// every portion from its state, which is the first's and those after it in order: 27 us and 53 in seven portions where the chain took 212.
// All entries' first portions come before their second ones, so that whole portions are dealt evenly and the short last ones behind them.
// Entries that more than fill the chip are taken longest first, heads beside each other, so that no long one is left for the end: eight documents of up to 2048 tokens, 64 heads of 128 x 64,
// 649 us a launch with the entries beside each other, 436 now.  (Where all run at once there is nothing to order, and finding the ranks is 1 us: sixteen entries of 200 tokens 27 and 28.)
enum { SSD_WHOLE = 0, SSD_STATES = 1, SSD_PORTIONS = 2 };
constexpr size_t ssd_state_elems(int NW) { return (size_t)NW * 16 * 256 + 4; }      // a workgroup's accumulators as it holds them, and the portion's decay
// the entry of rank r by its tokens, longest first (the entry r itself where there are more than 64)
__device__ __forceinline__ int entry_by_length(const StepMeta& m, int entries, int r) {
  if (entries > 64) return r;
  const int lane = threadIdx.x & 63, mine = lane < entries ? m.ent_count[lane] : -1;
  int rank = 0;
  for (int j = 0; j < entries; j++) { const int other = __builtin_amdgcn_readlane(mine, j); rank += other > mine || (other == mine && j < lane); }
  return __builtin_ctzll(__ballot(lane < entries && rank == r));
}
template <int NW, bool NORM = false, int MODE = SSD_WHOLE>
__global__ __launch_bounds__(256, NW == 1 ? 2 : 1) void ssd_block_kernel(StepMeta m, SsdArgs a) {
  constexpr int Q = SSD_BLOCK;
  constexpr double LOG2E = 1.4426950408889634;
  __shared__ float s_x[2][Q][32];
  __shared__ double s_cs[2][Q];        // base-2 logarithms, summed from the block's start
  __shared__ float s_dt[2][Q], s_end[2][Q];      // dt_j, exp(cs_64 - cs_j) dt_j
  __shared__ float s_part[4][Q][33];
  const int P = MODE == SSD_WHOLE ? 1 : a.portions, entries = gridDim.z / P, part = MODE == SSD_WHOLE ? 0 : blockIdx.z / entries, tile = blockIdx.y, tiles = gridDim.y;
  const int e = MODE == SSD_WHOLE ? (a.ranked ? entry_by_length(m, entries, blockIdx.z) : blockIdx.z) : blockIdx.z - part * entries, h = blockIdx.x, e0 = tile * 32, tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5, l31 = lane & 31;
  const int start = m.ent_start[e], cnt = m.ent_count[e], slot = m.ent_row[e], grp = h / (a.heads / a.groups);
  const int nblk = (cnt + Q - 1) / Q, b0 = MODE == SSD_WHOLE ? 0 : part * a.portion, b1 = MODE == SSD_WHOLE ? nblk : min(nblk, b0 + a.portion);
  if (MODE == SSD_STATES ? b1 >= nblk : b0 >= nblk) return;      // (the states of the last portion are nobody's start)
  const bool fresh = m.tok_pos[start] == 0;
  const bool ones = NORM && tile + 1 == tiles;
  const int ld = (int)a.ld, ldg = (int)a.ldgate, oX = a.x0 + h * a.E + e0, oB = a.b0 + grp * a.N, oC = a.c0 + grp * a.N;
  const float* base = a.row + (size_t)start * ld;
  const float* gbase = a.gates + (size_t)start * ldg + h;
  const float* gram = a.gram + ((size_t)ssd_first_block(start, e) * a.groups + grp) * (Q * Q);
  float* Sg = a.S + ((size_t)slot * a.heads + h) * (size_t)a.N * a.E;
  const bool colok = ones ? l31 == 0 : e0 + l31 < a.E;
  const int xcol = colok ? l31 : 0, n0 = 32 * wv * NW;
  const size_t sn = ones ? 1 : a.E, sc = ones ? 0 : e0 + l31;
  float* Snew = Sg;
  if (ones) {
    const int par = m.ent_par[e];
    const size_t at = ((size_t)slot * a.heads + h) * a.N;
    Sg = a.norm_S + (size_t)par * a.norm_buf + at; Snew = a.norm_S + (size_t)(par ^ 1) * a.norm_buf + at;
  }
  f32x16 S[NW];
  // slot 0: the entry's own state, slot p + 1: what portion p leaves
  auto left = [&](int p) { return a.states + ((((size_t)e * P + p) * a.heads + h) * tiles + tile) * ssd_state_elems(NW); };
  if (MODE != SSD_PORTIONS || nblk <= a.portion) {
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int n = n0 + 32 * w + (r & 3) + 8 * (r >> 2) + 4 * half;
        S[w][r] = (!fresh && n < a.N && colok && (MODE != SSD_STATES || part == 0)) ? Sg[n * sn + sc] : 0.f;
        if (MODE == SSD_STATES && part == 0) left(0)[(w * 16 + r) * 256 + tid] = S[w][r];      // (the last portion may have replaced it before the first one looks)
      }
  } else {
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int r = 0; r < 16; r++) S[w][r] = left(min(part, 1))[(w * 16 + r) * 256 + tid];
    for (int p = 2; p <= part; p++) {
      const float* s = left(p);
      const float g = s[NW * 4096];
#pragma unroll
      for (int w = 0; w < NW; w++)
#pragma unroll
        for (int r = 0; r < 16; r++) S[w][r] = fmaf(S[w][r], g, s[(w * 16 + r) * 256 + tid]);
    }
  }
  auto at = [](const float* p, unsigned int bytes) -> const float* { return reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + bytes); };
  // byte offset of row t0 + k of a block with `left` rows, clamped to its last one (ld < 2^21 floats: the factors fit 24 bits); the constant k stays out of registers
  auto row_at = [](int t0, int k, int left, int ld) -> unsigned int { return (unsigned int)(4 * (__mul24(t0, ld) + __mul24(min(k, left - 1 - t0), ld))); };
  auto row_off = [&](int t0, int k, int left) -> unsigned int { return row_at(t0, k, left, ld); };
  float B[NW][32], x[8], dt = 0.f, la = 0.f;      // B[n][j]: j = kk + 32 half
  f32x4 C[NW][2][4], G[2][2];                     // C[i][n]: four channels at a time; the Gram rows of this wave's sixteen keys j = 16 wv + 8 half + 0 .. 7
  // (what stands in state rows beyond N is finite and meets a factor of zero)
  auto fetch_B = [&](int b, float (*B)[32]) {
    const float* p = base + (size_t)b * Q * ld + oB;
    const int left = cnt - b * Q;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const int n = min(n0 + 32 * w + l31, a.N - 1);
#pragma unroll
      for (int kk = 0; kk < 32; kk++) B[w][kk] = *at(p, row_off(32 * half, kk, left) + 4 * n);
    }
  };
  auto fetch_C = [&](int b) {
    const float* p = base + (size_t)b * Q * ld + oC;
    const int left = cnt - b * Q;
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int it = 0; it < 2; it++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int n = n0 + 32 * w + 8 * q + 4 * half;
          C[w][it][q] = *reinterpret_cast<const f32x4*>(at(p, row_off(l31, 32 * it, left) + 4 * min(n, a.N - 4)));
        }
  };
  auto fetch_G = [&](int b) {
    const float* p = gram + (size_t)b * a.groups * (Q * Q);
#pragma unroll
    for (int it = 0; it < 2; it++)
      if (16 * wv <= 32 * it + 31)
#pragma unroll
        for (int q = 0; q < 2; q++) G[it][q] = *reinterpret_cast<const f32x4*>(at(p, 4u * (unsigned int)((32 * it + l31) * Q + 16 * wv + 8 * half + 4 * q)));
  };
  auto fetch_x = [&](int b) {
    const float* p = base + (size_t)b * Q * ld;
    const int left = cnt - b * Q;
#pragma unroll
    for (int u = 0; u < 8; u++) x[u] = ones ? 1.f : *at(p, row_off(tid >> 5, 8 * u, left) + 4 * (oX + xcol));
    if (wv == 0 && !a.fixed) { const float* g = gbase + (size_t)b * Q * ldg; const unsigned int off = row_at(lane, 0, left, ldg); dt = *at(g + a.dt_col, off); la = *at(g + a.log_col, off); }
  };
  auto stage = [&](int b) {
    const int buf = b & 1, left = cnt - b * Q;
#pragma unroll
    for (int u = 0; u < 8; u++) s_x[buf][(tid >> 5) + 8 * u][l31] = x[u];
    if (wv == 0) {
      double v = lane < left ? (double)la * LOG2E : 0.0;
      const float d = lane < left ? dt : 0.f;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) { const double p = __shfl_up(v, o, 64); if (lane >= o) v += p; }
      const double end = __shfl(v, 63, 64);
      s_cs[buf][lane] = v; s_dt[buf][lane] = d; s_end[buf][lane] = d * __builtin_amdgcn_exp2f((float)(end - v));
    }
  };
  if (a.fixed) { dt = a.dt0; la = a.fixed[a.heads + h]; }
  const float Dh = a.skip ? a.skip[h] : 0.f;
  auto add_block = [&](int buf, float (*B)[32]) {      // S = exp(cs_64) S + sum_j B_j (exp(cs_64 - cs_j) dt_j x_j)^T
    const float ge = __builtin_amdgcn_exp2f((float)s_cs[buf][Q - 1]);
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int r = 0; r < 16; r++) S[w][r] *= ge;
    if (n0 < a.N)
#pragma unroll
      for (int kk = 0; kk < 32; kk++) {
        const int j = kk + 32 * half;
        const float xs = s_x[buf][j][l31] * s_end[buf][j];
#pragma unroll
        for (int w = 0; w < NW; w++) S[w] = __builtin_amdgcn_mfma_f32_32x32x2f32(B[w][kk], xs, S[w], 0, 0, 0);
      }
  };
  fetch_x(b0);
  if constexpr (MODE == SSD_STATES) {
    double decay = 0.0;
    auto block = [&](int b, float (*now)[32], float (*next)[32]) {
      const bool more = b + 1 < b1;
      __syncthreads();      // the block's columns and sums stand; those of the block before have been read
      if (more) { fetch_x(b + 1); fetch_B(b + 1, next); }
      __builtin_amdgcn_sched_barrier(0);
      decay += s_cs[b & 1][Q - 1];
      add_block(b & 1, now);
      __builtin_amdgcn_sched_barrier(0);
      if (more) stage(b + 1);
      return more;
    };
    float B2[NW][32];
    fetch_B(b0, B);
    stage(b0);
    for (int b = b0; block(b, B, B2) && block(b + 1, B2, B); b += 2) {}
    float* s = left(part + 1);
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
      for (int r = 0; r < 16; r++) s[(w * 16 + r) * 256 + tid] = S[w][r];
    if (tid == 0) s[NW * 4096] = __builtin_amdgcn_exp2f((float)decay);
    return;
  }
  fetch_C(b0); fetch_G(b0);
  stage(b0);
  for (int b = b0; b < b1; b++) {
    const int buf = b & 1, t0 = b * Q;
    const bool more = b + 1 < b1;
    __syncthreads();      // the block's columns and sums stand; the shares of the block before have been read
    fetch_B(b, B);
    if (more) fetch_x(b + 1);
    __builtin_amdgcn_sched_barrier(0);      // (the phases stay apart: operands of a later one must not take registers early)
    f32x16 acc[2];
#pragma unroll
    for (int it = 0; it < 2; it++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[it][r] = 0.f;
    double csi[2];
    float ei[2];
#pragma unroll
    for (int it = 0; it < 2; it++) { csi[it] = s_cs[buf][32 * it + l31]; ei[it] = __builtin_amdgcn_exp2f((float)csi[it]); }
    // exp(cs_i) S_in^T C_i over this wave's state rows
#pragma unroll
    for (int w = 0; w < NW; w++)
      if (n0 + 32 * w < a.N)      // (wave-uniform)
#pragma unroll
        for (int r = 0; r < 16; r++) {
          const bool in = n0 + 32 * w + 8 * (r >> 2) + 4 * half < a.N;
#pragma unroll
          for (int it = 0; it < 2; it++) acc[it] = __builtin_amdgcn_mfma_f32_32x32x2f32(C[w][it][r >> 2][r & 3] * (in ? ei[it] : 0.f), S[w][r], acc[it], 0, 0, 0);
        }
    if (more) fetch_C(b + 1);
    __builtin_amdgcn_sched_barrier(0);
    // the block's own tokens: this wave's sixteen keys
    int ahead = l31 - 16 * wv - 8 * half;      // key k of this lane lies ahead of row 32 it + l31 when k > ahead + 32 it
    asm volatile("" : "+v"(ahead));            // (not hoisted into sixteen lane masks)
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int j = 16 * wv + 8 * half + k;
      const double csj = s_cs[buf][j];
      const float xj = s_x[buf][j][l31] * s_dt[buf][j];
#pragma unroll
      for (int it = 0; it < 2; it++) {
        // (for two of the waves all keys lie ahead of the first 32 rows: they multiply zeros while the others, whom they would wait for, do not)
        const float mij = k <= ahead + 32 * it ? G[it][k >> 2][k & 3] * __builtin_amdgcn_exp2f((float)(csi[it] - csj)) : 0.f;
        acc[it] = __builtin_amdgcn_mfma_f32_32x32x2f32(mij, xj, acc[it], 0, 0, 0);
      }
    }
    if (more) fetch_G(b + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int it = 0; it < 2; it++)
#pragma unroll
      for (int r = 0; r < 16; r++) s_part[wv][32 * it + (r & 3) + 8 * (r >> 2) + 4 * half][l31] = acc[it][r];
    __builtin_amdgcn_sched_barrier(0);
    add_block(buf, B);
    __builtin_amdgcn_sched_barrier(0);
    if (more) stage(b + 1);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int t = (tid >> 5) + 8 * u;
      if (t0 + t < cnt && colok)
        *(ones ? a.norm_out + (size_t)(start + t0 + t) * a.ldn + h : a.out + (size_t)(start + t0 + t) * a.ldo + h * a.E + e0 + l31) = fmaf(Dh, s_x[buf][t][l31], s_part[0][t][l31] + s_part[1][t][l31] + s_part[2][t][l31] + s_part[3][t][l31]);
    }
  }
  if (b1 < nblk) return;
#pragma unroll
  for (int w = 0; w < NW; w++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int n = n0 + 32 * w + (r & 3) + 8 * (r >> 2) + 4 * half;
      if (n < a.N && colok) Snew[n * sn + sc] = S[w][r];
    }
}

// The gates of a matrix memory in that form.  With the running maximum m_t = max(f_t + m_(t-1), i_t) of the log gates, the memory decays by exp(f_t + m_(t-1) - m_t), takes
// k v^T by exp(i_t - m_t), and divides by at least exp(-m_t).  A token is the map m -> max(f + m, i), and such maps compose to maps of the same form, so a scan over lanes,
// waves and portions of 1024 tokens gives every m_t from sums of the f alone (no difference of two long sums).  The maxima are kept in double: a thread takes the maximum
// before its tokens from the composed maps and its neighbour's from its own steps, and in fp32 the two differed by a rounding, which is a factor on the whole memory.  The
// maximum that the entry leaves is an fp32 number, so its last token's is rounded to that before its gates are made.  2048 tokens, 8 heads of 128 x 256: token by token 940 us a layer,
// bound by each token's dependent step; 80 in blocks, their chain of 32 in seven portions.  Grid: (entries, heads).
struct GateScanArgs {
  const float* proj; long long ldp; int i0, f0;      // the columns of the log gates
  float* mx; size_t mx_buf;                          // [2][slots][heads]
  float* gates; int heads;                           // [T][take (heads) | log decay (heads) | exp(-m) (heads)]
};
template <int TPT = 4>      // tokens of a thread
__global__ __launch_bounds__(256) void gate_scan_kernel(StepMeta m, GateScanArgs a) {
  __shared__ double s_f[2][4], s_m[2][4];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int start = m.ent_start[e], cnt = m.ent_count[e], row = m.ent_row[e], par = m.ent_par[e];
  double carry = m.tok_pos[start] == 0 ? 0.f : a.mx[(size_t)par * a.mx_buf + (size_t)row * a.heads + h];
  for (int t0 = 0, p = 0; t0 < cnt; t0 += 256 * TPT, p ^= 1) {
    double f[TPT], ig[TPT];
#pragma unroll
    for (int u = 0; u < TPT; u++) {      // (past the end m -> max(0 + m, -inf))
      const int t = t0 + TPT * tid + u;
      const float* r = a.proj + (size_t)(start + min(t, cnt - 1)) * a.ldp;
      const float fv = r[a.f0 + h], iv = r[a.i0 + h];
      f[u] = t < cnt ? fv : 0.f; ig[u] = t < cnt ? iv : -INFINITY;
    }
    double F = f[0], M = ig[0];
#pragma unroll
    for (int u = 1; u < TPT; u++) { M = fmax(M + f[u], ig[u]); F += f[u]; }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double pf = __shfl_up(F, o, 64), pm = __shfl_up(M, o, 64);
      if (lane >= o) { M = fmax(pm + F, M); F += pf; }
    }
    if (lane == 63) { s_f[p][wv] = F; s_m[p][wv] = M; }
    const double bf = __shfl_up(F, 1, 64), bm = __shfl_up(M, 1, 64);      // the map of the lanes before
    __syncthreads();      // (two buffers: the next portion's sums are written before all have read these)
    double before = carry;
#pragma unroll
    for (int w = 0; w < 4; w++) { if (w < wv) before = fmax(before + s_f[p][w], s_m[p][w]); carry = fmax(carry + s_f[p][w], s_m[p][w]); }
    if (lane > 0) before = fmax(before + bf, bm);
#pragma unroll
    for (int u = 0; u < TPT; u++) {
      const int t = t0 + TPT * tid + u;
      double now = fmax(before + f[u], ig[u]);
      if (t == cnt - 1) now = (float)now;
      if (t < cnt) {
        float* o = a.gates + (size_t)(start + t) * 3 * a.heads + h;
        const float mf = (float)now;
        o[0] = expf((float)(ig[u] - now)); o[a.heads] = (float)(f[u] + before - now); o[2 * a.heads] = expf(-mf) * (1.0f + (float)(mf - now));      // exp(-now), now = mf + what its rounding left
      }
      before = now;
    }
  }
  if (tid == 0) a.mx[(size_t)(par ^ 1) * a.mx_buf + (size_t)row * a.heads + h] = (float)carry;
}

}  // namespace tgx
