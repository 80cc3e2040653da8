// stack_few.h — the products of layered models (stack_gemm.h) for A FEW rows: 3 to 64 activation rows, the tiles of sixteen rows of a grouped product with few
// (token, expert) pairs, and matrices of so few rows (a router's) that 64-wide tiles would stand empty.
//
// What bounds it: the weights cross once, so the stream of weight bytes is the floor; the vector form (stack_gemv_kernel, two columns a wave) instead moved every
// activation row through L2 for every two columns — eight rows of 4 KB for 4 KB of weights — and streamed the weights again for every tile of four or eight rows.
// Here a workgroup owns SIXTEEN columns and up to 64 rows, so an activation byte serves eight times as many weights and a weight byte is read once for all rows.  The
// products are v_mfma_f32_16x16x4_f32 on the stored weights widened to 32 bits and the activations as they are: nothing is rounded or split, as in the vector form
// (at sixteen rows the 32-bit rate costs less than the stream: 0.6 us for 3072 x 1024 on the whole chip).  Products are summed in runs of 32 (a half step), the runs of a step,
// the steps of a wave and the waves in chains of their own (fp32 logits of two layers of 1024 / 8192 channels against 64 bits, four / sixteen rows: 1.25 / 1.17 times the vector
// form's error with one chain over a wave's whole share of K, 0.95 / 0.97 so).
//
// The waves of a workgroup divide K in steps of 64 and have nothing to do with each other until their sums meet in LDS, in a fixed order (results do not depend on
// timing).  A step arrives by LDS-DMA in the wave's own ring: straight loads in the matrix operand's layout put sixteen rows under sixteen neighbouring lanes, one
// address lookup a lane — 26 us for 32000 x 1024 however many were in flight; a DMA piece covers whole lines (eight weight rows of 128 bytes, four activation rows of 256).
// LDS image: 16-byte chunk c of row r in slot c ^ (r & 7), applied on the global side and in the fragment reads (as in gemm_dma.h).
// The host picks waves and ring depth so that narrow matrices (N / 16 workgroups) have as much of K in flight at once as LDS holds.
// Any M, N; K a multiple of 8, 16-byte aligned rows (launch_gemm's condition).
//
// Measured against the vector form (us, medians of a step's launches, bf16): sixteen rows 2 x 3072 x 1024 19.0 -> 8.5, 32000 x 1024 82 -> 24; eight rows 2 x 8192 x 2048 35 -> 20,
// 2048 x 8192 26 -> 14; four rows 2 x 8192 x 2048 22.7 -> 19.8 (3.4 TB/s), 2048 x 8192 13.0 -> 14.2; against the 64-wide tiles, 47 rows: 2 x 3072 x 1024 27 -> 17, 1024 x 3072 42 -> 20.
#pragma once
#include "args_ahead.h"
#include "gemm_dma.h"
#include "stack_gemm.h"

namespace tgx {

constexpr int few_max_waves(int mb) { return mb == 1 ? 16 : 8; }      // 128 / 256 registers a wave

// XP: the pieces (four activation rows each) of a tile of sixteen that are brought: 1 or 2 where the step has no more than four or eight rows (the rest of the operand repeats them and is
// not stored).  A step of 64 k is 2 KB of weights and XP KB of activations, which cross from L2 for every sixteen columns.  us a launch, XP 4 -> as many as there are rows, four rows:
// 2304 x 1024 5.7 -> 5.1, 8192 x 1024 8.3 -> 7.2, 32000 x 1024 20.8 -> 17.8, 2 x 8192 x 2048 21.5 -> 18.6; eight: 2048 x 4096 11.6 -> 10.5, 8192 x 2048 13.3 -> 11.9, 2048 x 8192
// 18.8 -> 16.7, 32000 x 2048 35.0 -> 33.7
template <int DT, bool DUAL, int MB, int XP> constexpr int few_step_bytes() { return (DUAL ? 2 : 1) * (DT == DT_F32 ? 4096 : 2048) + MB * XP * 1024; }
// LDS of a workgroup: the waves' rings, which the sums use again at the end
template <int DT, bool DUAL, int MB, int XP> constexpr size_t few_lds_bytes(int waves, int depth) {
  const size_t ring = (size_t)waves * depth * few_step_bytes<DT, DUAL, MB, XP>(), sums = (size_t)waves * (DUAL ? 2 : 1) * MB * 1024;
  return ring > sums ? ring : sums;
}

// what a lane reads whose place lies past the end of K (the last step of a K that is no multiple of 64)
__device__ const u32x4 few_zeros = {0u, 0u, 0u, 0u};

template <int DT, int EPI, bool DUAL, int MB, int XP>
__device__ __forceinline__ void stack_few_body(const StackGemmArgs& a, const int depth, const int z, const int mbase, const int mend) {
  constexpr int NB = DUAL ? 2 : 1, WP = DT == DT_F32 ? 4 : 2;       // 1-KB pieces of a step's weight rows (per matrix)
  constexpr int PIECES = NB * WP + MB * XP, STEP = few_step_bytes<DT, DUAL, MB, XP>();
  static_assert(XP == 4 || MB == 1, "all rows of a tile but the only one");
  extern __shared__ __attribute__((aligned(1024))) unsigned char few_lds[];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
  const int li = lane & 15, q = lane >> 4;                          // row (column) of the operands, quarter of a half step's k
  const int n0 = blockIdx.x * 16, N = args_ahead(a.N, a, (int)blockDim.x), steps = (a.K + 63) >> 6;
  if (n0 >= N) return;                                            // (the narrower product of a pair)
  unsigned char* ring = few_lds + (size_t)wv * depth * STEP;
  const unsigned ring_lds = (unsigned)(size_t)ring;

  // DMA map: rows and slots of this lane in every piece; a slot past the end of K takes zeros
  const elem_t<DT>* wsrc[NB][WP];
  const float* xsrc[MB][XP];
  constexpr int WROWS = 16 / WP;                                    // weight rows per piece
  const int wslot = lane % (64 / WROWS), xslot = lane & 15;
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int p = 0; p < WP; p++)
      wsrc[b][p] = reinterpret_cast<const elem_t<DT>*>(b ? a.B2 : a.B) + (size_t)z * a.b_zstride + (size_t)min(n0 + p * WROWS + lane / (64 / WROWS), N - 1) * a.ldb;
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int p = 0; p < XP; p++) {
      const int mc = min(mbase + 16 * i + 4 * p + q, mend - 1);
      xsrc[i][p] = a.A + (size_t)z * a.a_zoff + (size_t)(a.a_rows ? a.a_rows[mc] : mc) * a.lda;
    }
  auto issue = [&](int c, int slot) {
    unsigned dst = ring_lds + (unsigned)(slot * STEP);
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int p = 0; p < WP; p++, dst += 1024) {
        const int row = p * WROWS + lane / (64 / WROWS), chunk = wslot ^ (row & 7);
        const int k = 64 * c + (DT == DT_F32 ? 4 : 8) * chunk;
        dma_1k(k < a.K ? (const void*)(wsrc[b][p] + k) : (const void*)&few_zeros, dst);
      }
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int p = 0; p < XP; p++, dst += 1024) {
        const int k = 64 * c + 4 * (xslot ^ ((4 * p + q) & 7));
        dma_1k(k < a.K ? (const void*)(xsrc[i][p] + k) : (const void*)&few_zeros, dst);
      }
  };
  // a step's sums, one set per half step (two chains of products in flight), are added to the wave's when the next step's operands have landed
  f32x4 acc[NB][MB], part[2][NB][MB];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int i = 0; i < MB; i++) acc[b][i] = part[0][b][i] = part[1][b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto collect = [&] {
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int i = 0; i < MB; i++) acc[b][i] += part[0][b][i] + part[1][b][i];
  };
  auto product = [&](int slot, auto R16) {                          // R16: activations rounded to the storage type first (option act.round16)
    const unsigned char* st = ring + slot * STEP;
    collect();
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int i = 0; i < MB; i++) part[h][b][i] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int sl = 4 * h + q;                                     // this lane's slice of the step
      float w[NB][8];
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const unsigned char* rb = st + b * WP * 1024;
        Slice8<DT> s;
        if constexpr (DT == DT_F32) {
          s.v = *reinterpret_cast<const u32x4*>(rb + li * 256 + (((2 * sl) ^ (li & 7)) << 4));
          s.w = *reinterpret_cast<const u32x4*>(rb + li * 256 + (((2 * sl + 1) ^ (li & 7)) << 4));
        } else s.v = *reinterpret_cast<const u32x4*>(rb + li * 128 + ((sl ^ (li & 7)) << 4));
        slice_unpack<DT>(s, w[b]);
      }
#pragma unroll
      for (int i = 0; i < MB; i++) {
        const int xr = li & (4 * XP - 1);
        const unsigned char* rx = st + NB * WP * 1024 + i * 4096 + xr * 256;
        const f32x4 x0 = *reinterpret_cast<const f32x4*>(rx + (((2 * sl) ^ (xr & 7)) << 4)), x1 = *reinterpret_cast<const f32x4*>(rx + (((2 * sl + 1) ^ (xr & 7)) << 4));
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float v = e < 4 ? x0[e & 3] : x1[e & 3], x = R16.value ? round_storage_if<DT>(v, 1) : v;
#pragma unroll
          for (int b = 0; b < NB; b++) part[h][b][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, w[b][e], part[h][b][i], 0, 0, 0);
        }
      }
    }
  };
  const int mine = wv < steps ? (steps - wv + nw - 1) / nw : 0;     // this wave's steps: wv, wv + nw, ..
  for (int i = 0; i < min(depth, mine); i++) issue(wv + i * nw, i);
  for (int i = 0, slot = 0; i < mine; i++) {
    // step i has landed once only the pieces of the steps issued behind it may fly (DMA completes in order)
    const int later = min(depth - 1, mine - 1 - i);
    if (later >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PIECES) : "memory");
    else if (later == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PIECES) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (a.terms == 1) product(slot, std::true_type{}); else product(slot, std::false_type{});
    if (i + depth < mine) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // this wave's reads of the slot are done
      issue(wv + (i + depth) * nw, slot);
    }
    slot = slot + 1 == depth ? 0 : slot + 1;
  }

  collect();
  __syncthreads();                                                  // every wave is done with its ring
  float* red = reinterpret_cast<float*>(few_lds);                   // [waves][NB * MB * 4][64]
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) red[((wv * NB + b) * MB * 4 + i * 4 + r) * 64 + lane] = acc[b][i][r];
  __syncthreads();
  // C layout of the 16 x 16 product: column = lane & 15, row = 4 (lane >> 4) + r
  for (int o = threadIdx.x; o < MB * 256; o += blockDim.x) {
    const int l = o & 63, ir = o >> 6, m = mbase + (ir >> 2) * 16 + 4 * (l >> 4) + (ir & 3), n = n0 + (l & 15);
    if (m >= mend || n >= a.N) continue;
    auto total = [&](auto WAVES, int b) {                           // (all on their way at once)
      constexpr int W = decltype(WAVES)::value;
      float t[W], s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < W; w++) t[w] = red[((min(w, nw - 1) * NB + b) * MB * 4 + ir) * 64 + l];
#pragma unroll
      for (int w = 0; w < W; w++) s[w & 3] += w < nw ? t[w] : 0.f;
      return (s[0] + s[1]) + (s[2] + s[3]);
    };
    float v[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
      v[b] = nw == 1   ? total(std::integral_constant<int, 1>{}, b)
             : nw <= 4 ? total(std::integral_constant<int, 4>{}, b)
             : nw <= 8 ? total(std::integral_constant<int, 8>{}, b)
                       : total(std::integral_constant<int, few_max_waves(MB)>{}, b);
    sg_finish<EPI>(a, z, m, n, v[0], v[NB - 1]);
  }
}

template <int DT, int EPI, bool DUAL, int MB, int XP>
__global__ __launch_bounds__(64 * few_max_waves(MB)) void stack_few_kernel(const StackGemmArgs a, const int depth) {
  int z = blockIdx.z, m0 = blockIdx.y * 16 * MB, rows_end = a.M;
  if (args_ahead(a.z_off, a, (int)blockDim.x)) {
    if ((int)blockIdx.y >= *a.n_tiles) return;
    z = a.tile_z[blockIdx.y]; m0 = a.tile_m0[blockIdx.y]; rows_end = a.z_off[z + 1];
  }
  stack_few_body<DT, EPI, DUAL, MB, XP>(a, depth, z, m0, min(rows_end, m0 + 16 * MB));
}
// two products that do not need each other, of the same rows and contraction length, in one launch: blockIdx.z chooses (the low-rank pair of a channel-delta layer, sixteen rows of
// 1024 x 128 each: 4.7 us and 4.7, 5.7 together)
template <int DT, int MB, int XP>
__global__ __launch_bounds__(64 * few_max_waves(MB)) void stack_few_pair_kernel(const StackGemmArgs a, const StackGemmArgs b, const int depth) {
  if (blockIdx.z == 0) stack_few_body<DT, SG_STORE, false, MB, XP>(a, depth, 0, 0, a.M);      // (one tile of rows)
  else stack_few_body<DT, SG_STORE, false, MB, XP>(b, depth, 0, 0, b.M);
}

// pieces of four activation rows that the tiles of sixteen need (a plan's rows are counted on the device)
inline int few_pieces(const StackGemmArgs& a) { return a.z_off || a.M > 8 ? 4 : a.M > 4 ? 2 : 1; }
// Waves and ring depth: some eight waves a compute unit (2048 on the chip) and four a workgroup at least, never more than K has steps; two steps of each in flight, one
// where the launch has a thousand workgroups that cover for each other.  Measured, us at waves / depth 4/1, 4/2, 8/1, 8/2, 16/1: sixteen rows 1024 x 1024 (64 workgroups):
// 6.7, 5.9, 5.6, 5.6, 5.5; eight rows 2048 x 8192 (128): 36.6, 22.7, 23.3, 18.5, 18.8; 4096 x 2048 (256): 12.8, 9.3, 9.8, 8.8, 9.3; 8192 x 2048 (512): 15.1, 13.0, 14.0, 15.5,
// 15.7; sixteen rows 24576 x 1024 (1536): 16.8, 17.7, 18.1, 26.7, 26.8
struct FewPlan { int nw, depth; size_t lds; };
template <int DT, bool DUAL, int MB, int XP>
inline FewPlan few_plan(int num_cus, long long wgs, int K) {
  const int steps = (K + 63) / 64;
  FewPlan p{4, 1, 0};
  while (p.nw < few_max_waves(MB) && wgs * p.nw < 8LL * num_cus) p.nw *= 2;
  while (p.nw > 1 && p.nw > steps) p.nw /= 2;
  p.depth = wgs >= 4LL * num_cus || p.nw >= steps ? 1 : 2;
  while ((p.lds = few_lds_bytes<DT, DUAL, MB, XP>(p.nw, p.depth)) > 160 * 1024) { if (p.depth > 1) p.depth--; else p.nw /= 2; }
  return p;
}

}  // namespace tgx
