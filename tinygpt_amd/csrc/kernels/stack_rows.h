// stack_rows.h — the products of layered models (stack_gemm.h) for the (token, expert) pairs of a step of few tokens, up to 128, grouped by expert in the kernel itself.  Made for a few
// rows an expert: up to six on average (stack.hip sends more to a plan and sixteen-row tiles).
//
// What bounds it: the weights of a chosen expert cross once for every eight rows that it has, so as a rule once (25 MB for four tokens of 1024 channels and two of eight experts of 1536: 4 us at the rate of a large read); beside
// that stand a launch and whatever chain of loads comes before the first weight.  The form before it (moe_plan_kernel, then stack_few_kernel on sixteen-row tiles) paid a launch
// for the plan, four dependent loads (number of tiles, tile, rows, activations) in each product, sixteen rows of activations for the one to four that an expert has and
// sixteen-row matrix instructions for them.  Here every workgroup reads the choices themselves (one load, two ballots), and the products are v_mfma_f32_4x4x1_f32 in
// sixteen blocks: a block is a slice of eight k, its four rows are activations and its four columns weights, so a tile of four rows costs a quarter of the 16 x 16 form's
// matrix time and the weights need no staging: sixteen lanes read 256 bytes of one row (whole lines), four rows a load, straight into the operand's registers.
// Nothing is rounded or split.  A block sums its own slices (eight products a chunk of 128 k), blocks and waves meet in a fixed order at the end.
//
// Rows of an expert in tiles of eight, sixteen columns of one matrix or eight of two a workgroup, K in chunks of 128 that the waves divide, two of a wave's on their way.  A wave's own
// instructions are what is left beside the stream (four cycles each, three waves a SIMD): so a wave is given several chunks (two waves a workgroup where that fills the chip),
// loads none past its last, and its sixteen blocks' sums meet in LDS as vectors and not lane by lane.
//
// Measured, us a launch in a row of them over different weights, bf16, here (before, from a step's trace: plan 2.8 beside each pair): sixteen tokens, two of eight experts and a shared
// one, 1536 x 1024 12.1 (13.8), 1024 x 1536 11.5 (12.9); four tokens, two of eight, 2 x 1536 x 1024 10.8 (14.6), 1024 x 1536 7.4 (9.6); one token, four of sixteen,
// 2 x 2048 x 2048 15.6 (18.4; 4.3 TB/s), 2048 x 2048 10.0 (11.3).
// Any N and pairs; K a multiple of 8, 16-byte aligned rows (launch_gemm's condition).
#pragma once
#include "args_ahead.h"
#include "stack_gemm.h"

namespace tgx {

constexpr int ROWS_MAX_WAVES = 4;
constexpr int ROWS_TILE = 8;
constexpr int rows_cols(bool dual) { return dual ? 8 : 16; }
constexpr int ROWS_SUM_ROWS = 8 * 68;      // vectors of four of a wave's sums
constexpr size_t rows_lds(int waves) { return (size_t)waves * ROWS_SUM_ROWS * 16; }

template <int DT, int EPI, bool DUAL>
__global__ __launch_bounds__(64 * ROWS_MAX_WAVES, 3) void stack_rows_kernel(const StackGemmArgs a) {
  constexpr int NB = DUAL ? 2 : 1, RT = ROWS_TILE, COLS = rows_cols(DUAL), NG = COLS / 4;
  __shared__ int s_pair[ROWS_MAX_PAIRS];
  extern __shared__ __attribute__((aligned(16))) float s_sum[];     // rows_lds()
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  // the pairs of this workgroup's expert: blockIdx.y is the expert, or, where there are fewer pairs than experts, a pair that stands for its expert if none before it does
  const int n_pairs = args_ahead(a.n_pairs, a, (int)blockDim.x);
  const int c0 = lane < n_pairs ? a.sel[lane] : -1, c1 = lane + 64 < n_pairs ? a.sel[lane + 64] : -1;
  const bool by_pair = n_pairs < a.experts;
  const int y = blockIdx.y, z = by_pair ? __builtin_amdgcn_readlane(y < 64 ? c0 : c1, y & 63) : y;
  if (z >= a.experts) return;                                       // (an identity output: no product)
  const unsigned long long m0 = __ballot(c0 == z), m1 = __ballot(c1 == z);
  if (by_pair && (m0 ? __builtin_ctzll(m0) : 64 + __builtin_ctzll(m1)) != y) return;
  const int rows = __builtin_popcountll(m0) + __builtin_popcountll(m1);
  if ((int)blockIdx.z * RT >= rows) return;
  const unsigned long long below = (1ull << lane) - 1ull;
  if (wv == 0) {
    if (c0 == z) s_pair[__builtin_popcountll(m0 & below)] = lane;
    if (c1 == z) s_pair[__builtin_popcountll(m0) + __builtin_popcountll(m1 & below)] = lane + 64;
  }
  __syncthreads();
  const int n0 = blockIdx.x * COLS, nsl = a.K >> 3, chunks = (nsl + 15) >> 4;
  const int j = lane & 3, bl = lane >> 2;                           // row (column) of the lane's block, and the block: a slice of eight k

  // a column's row of weights: a scalar base and the lane's offset (COLS rows of K elements fit 32 bits for any K below 2^28)
  const elem_t<DT>* wbase[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) wbase[b] = reinterpret_cast<const elem_t<DT>*>(b ? a.B2 : a.B) + (size_t)z * a.b_zstride + (size_t)n0 * a.ldb;
  unsigned woff[NG];
#pragma unroll
  for (int g = 0; g < NG; g++) woff[g] = (unsigned)min(4 * g + j, a.N - 1 - n0) * (unsigned)a.ldb;

  auto body = [&](auto RSc, int r0, int here) {
    constexpr int RS = decltype(RSc)::value;
    const float* xrow[RS];
#pragma unroll
    for (int s = 0; s < RS; s++) xrow[s] = a.A + (size_t)(s_pair[r0 + min(4 * s + j, here - 1)] / a.pairs_per_row) * a.lda;
    struct Buf { Slice8<DT> w[NB][NG]; f32x4 x[RS][2]; };
    auto load = [&](Buf& f, int c) {                                // (past the end of K: the last slice again, dropped in product)
      const unsigned k = 8u * (unsigned)min(16 * c + bl, nsl - 1);
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int g = 0; g < NG; g++) f.w[b][g] = load_slice_nt<DT>(wbase[b] + (woff[g] + k), 0);
#pragma unroll
      for (int s = 0; s < RS; s++) {
        const f32x4* xp = reinterpret_cast<const f32x4*>(xrow[s] + k);
        f.x[s][0] = xp[0]; f.x[s][1] = xp[1];
      }
    };
    f32x4 acc[NB][RS][NG];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int s = 0; s < RS; s++)
#pragma unroll
        for (int g = 0; g < NG; g++) acc[b][s][g] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto product = [&](Buf& f, int c) {
      if (16 * c + 16 > nsl && 16 * c + bl >= nsl) {
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int g = 0; g < NG; g++) f.w[b][g] = Slice8<DT>{};
#pragma unroll
        for (int s = 0; s < RS; s++) f.x[s][0] = f.x[s][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      if (a.terms == 1) {
#pragma unroll
        for (int s = 0; s < RS; s++)
#pragma unroll
          for (int e = 0; e < 8; e++) f.x[s][e >> 2][e & 3] = round_storage_if<DT>(f.x[s][e >> 2][e & 3], 1);
      }
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int g = 0; g < NG; g += 2) {
          float w[2][8];
          slice_unpack<DT>(f.w[b][g], w[0]);
          slice_unpack<DT>(f.w[b][g + 1], w[1]);
#pragma unroll
          for (int e = 0; e < 8; e++)
#pragma unroll
            for (int s = 0; s < RS; s++)
#pragma unroll
              for (int i = 0; i < 2; i++) acc[b][s][g + i] = __builtin_amdgcn_mfma_f32_4x4x1f32(f.x[s][e >> 2][e & 3], w[i][e], acc[b][s][g + i], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);                        // (eight registers of widened weights a group, not all of them at once)
        }
    };
    // this wave's chunks wv, wv + nw, ..: two on their way, none past the last
    const int mine = wv < chunks ? (chunks - 1 - wv) / nw + 1 : 0;
    Buf f0, f1;
    int c = wv, i = 0;
    if (mine > 0) load(f0, c);
#pragma unroll 1
    for (; i + 2 < mine; i += 2, c += 2 * nw) {
      load(f1, c + nw);
      product(f0, c);
      load(f0, c + 2 * nw);
      product(f1, c + nw);
    }
    if (mine - i == 2) { load(f1, c + nw); product(f0, c); f0 = f1; c += nw; }
    if (mine > 0) product(f0, c);
    // the sums of the sixteen blocks meet in the wave's own LDS: a lane adds up four rows of one column, over all blocks or the share of them that the wave has lanes for
    constexpr int SETS = NB * RS * NG, PARTS = 16 / SETS;           // (4 SETS columns of four rows)
    f32x4* mine4 = reinterpret_cast<f32x4*>(s_sum) + (size_t)wv * ROWS_SUM_ROWS;
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int s = 0; s < RS; s++)
#pragma unroll
        for (int g = 0; g < NG; g++) mine4[((b * RS + s) * NG + g) * 68 + lane] = acc[b][s][g];      // (rows of 68: the columns' reads fall into other banks)
    wave_fence();
    const int set = (lane >> 2) % SETS, part = lane / (4 * SETS);
    f32x4 v = mine4[set * 68 + j + 4 * part];
#pragma unroll
    for (int i = PARTS; i < 16; i += PARTS) v += mine4[set * 68 + j + 4 * (part + i)];
#pragma unroll
    for (int o = 4 * SETS; o < 64; o *= 2)
#pragma unroll
      for (int r = 0; r < 4; r++) v[r] += __shfl_xor(v[r], o, 64);
    wave_fence();
    if (part == 0) mine4[lane] = v;                                 // [matrix][four rows][column]
  };
  // (a token chooses an expert once, so the grid's tiles hold all of an expert's pairs; where scores that are no numbers let it choose one again, a workgroup goes on to the next)
  for (int r0 = blockIdx.z * RT; r0 < rows; r0 += gridDim.z * RT) {
    const int here = min(RT, rows - r0);
    if (here <= 4) body(std::integral_constant<int, 1>{}, r0, here);
    else if constexpr (RT > 4) body(std::integral_constant<int, 2>{}, r0, here);
    __syncthreads();
    const int rs = here <= 4 ? 1 : 2;
    for (int o = threadIdx.x; o < here * COLS; o += blockDim.x) {
      const int r = o / COLS, n = n0 + o % COLS;
      if (n >= a.N) continue;
      float v[NB];
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const float* p = s_sum + 4 * ((b * rs + (r >> 2)) * COLS + o % COLS) + (r & 3);
        v[b] = p[0];
        for (int w = 1; w < nw; w++) v[b] += p[(size_t)w * ROWS_SUM_ROWS * 4];
      }
      sg_finish<EPI>(a, z, s_pair[r0 + r], n, v[0], v[NB - 1]);
    }
    __syncthreads();
  }
}

}  // namespace tgx
