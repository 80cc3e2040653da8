// stack_line.h — the products of layered models (stack_gemm.h) for prompts, 16-bit storage: both operands by LDS-DMA in whole 128-byte lines.
//
// What bounded them: stack_gemm_kernel brings every operand byte through registers (fp32 activations split into two 16-bit terms by every column tile again) with two
// barriers a step, on 64 x 64 or 128 x 128 tiles: 0.65 PFLOP/s executed on 11264 x 8192 x 2048, where the flat families' kernels reach 1.2.  Here the activations are split
// ONCE into lines [row][K / 32][32 first terms | 32 second terms] (split_terms_kernel, the norm in front, or the epilogue of the product in front), so that the two terms of a k32 block are one
// line, weights come as whole k64 lines, and the tiles are those of gemm_dma.h:
//   256 x 256, eight waves of 64 x 128, a ring of five 32-KB units (gemm_dma8i_kernel's schedule): products that fill the chip with such tiles
//   128 x 128, eight waves = two row halves x the four k16 steps of a stage, or quadrants x two of them, a ring of three 48-KB stages (gemm_dma8k_kernel's): the others
// The products of one output are summed in the same two-term form as before (small term first); only the order of the fp32 sums differs.
// Dual products (gate and up) take their two matrices in alternate blocks of 32 columns of a tile, so that both values of an output meet in one lane.
// A last round of tiles that is at most half full is halved over K (SHARED, line_plan.h); not in grouped products, whose plan deals an expert's rows to its tiles in any order: a row
// would be summed whole in one pass and in halves in the next.
// Tiles are dealt to the XCDs in contiguous runs, each run walked eight row tiles at a time: an XCD's workgroups share row blocks and weight tiles in its L2.
#pragma once
#include "../line_plan.h"
#include "gemm_dma.h"
#include "stack_gemm.h"

namespace tgx {

struct LineArgs {
  StackGemmArgs g;                      // A is not read: the terms are
  const bf16_t* terms; long long ldt;   // [rows][ldt]: interleaved lines; batch member z starts z * 2 * a_zoff elements into a row
  int gm, gn;                           // row and column tiles (gm: upper bound for grouped products)
  int cus;                              // SHARED: the last tiles are halved over K (line_plan.h, rounds of cus workgroups); [halved tile][2] who has come and whose sums lie ready
  int* met; float* sums;                // (zero between launches), and the sums
};

constexpr size_t LINE256_LDS = 5 * 32 * 1024, LINE128_LDS = 3 * 48 * 1024;

// one workgroup per row: fp32 [rows][lda] -> lines of two 16-bit terms, `cols` of them (a multiple of 32); mode 1 (option act.round16): the rounded first term alone
template <int DT>
__global__ __launch_bounds__(256) void split_terms_kernel(const float* a, long long lda, int cols, int one_term, bf16_t* out) {
  const float* src = a + (size_t)blockIdx.x * lda;
  bf16_t* dst = out + (size_t)blockIdx.x * 2 * cols;
  for (int c = 8 * threadIdx.x; c < cols; c += 2048) {
    const f32x4 x0 = *reinterpret_cast<const f32x4*>(src + c), x1 = *reinterpret_cast<const f32x4*>(src + c + 4);
    u32x4 h, l;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const float u = t < 2 ? x0[2 * t] : x1[2 * t - 4], v = t < 2 ? x0[2 * t + 1] : x1[2 * t - 3];
      bf16_t hu, lu, hv, lv;
      split16<DT>(u, hu, lu);
      split16<DT>(v, hv, lv);
      h[t] = (unsigned int)hu | ((unsigned int)hv << 16);
      l[t] = one_term ? 0u : (unsigned int)lu | ((unsigned int)lv << 16);
    }
    bf16_t* line = dst + (size_t)(c >> 5) * 64 + (c & 31);
    *reinterpret_cast<u32x4*>(line) = h;
    *reinterpret_cast<u32x4*>(line + 32) = l;
  }
}

// tile t in bands of eight row tiles
__device__ __forceinline__ void line_at(int t, int gm, int gn, int& tm, int& tn) {
  const int band = t / (8 * gn), rows = min(8, gm - 8 * band), in = t - band * 8 * gn;
  tm = 8 * band + in % rows;
  tn = in / rows;
}
// the id-th of `total` workgroups to its tile: runs of consecutive tiles per XCD (workgroup ids mod 8)
__device__ __forceinline__ int line_run(int id, int total) { return (id & 7) * (total >> 3) + min(id & 7, total & 7) + (id >> 3); }

// rows of the tile and where its operands lie
struct LineTile { int z, mbase, mend, tn, k0, nk, rest; };      // its steps of 64 from k0 on; the number of a halved one (-1: whole)
template <bool SHARED>
__device__ __forceinline__ bool line_place(const LineArgs& a, int TM, LineTile& t) {
  int tm;
  const int id = (int)blockIdx.x, gm = !SHARED && a.g.z_off ? min(a.gm, *a.g.n_tiles) : a.gm, nk = a.g.K >> 6;
  const LineShare sh = SHARED ? line_share(gm * a.gn, TM, nk, a.cus) : LineShare{gm * a.gn, 0};
  t.k0 = 0; t.nk = nk; t.rest = -1;
  if (id < sh.whole) line_at(line_run(id, sh.whole), gm, a.gn, tm, t.tn);
  else if (!SHARED || id >= sh.whole + 2 * sh.rest) return false;
  else {      // first halves of all, then the second ones: neighbours share operands in an XCD's L2
    const int at = id - sh.whole, half = at >= sh.rest;
    t.rest = line_run(half ? at - sh.rest : at, sh.rest);
    line_at(sh.whole + t.rest, gm, a.gn, tm, t.tn);
    t.k0 = half ? nk >> 1 : 0;
    t.nk = half ? nk - t.k0 : nk >> 1;
  }
  if (!SHARED && a.g.z_off) { t.z = a.g.tile_z[tm]; t.mbase = a.g.tile_m0[tm]; t.mend = min(a.g.z_off[t.z + 1], t.mbase + TM); }
  else { t.z = blockIdx.y; t.mbase = tm * TM; t.mend = min(a.g.M, t.mbase + TM); }
  return true;
}
// A halved tile's workgroups meet in memory: the first to have its sums writes them (numbers in pairs, past the L2 of its XCD, which the other's does not see) and is done; the
// second adds them to its own, whichever half that is, and goes on to the epilogue.  What it waits for at most is the first one's writes, which nothing holds up.
__device__ __forceinline__ void line_give(float* at, float x, float y) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(at), (unsigned long long)__float_as_uint(x) | ((unsigned long long)__float_as_uint(y) << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
typedef __attribute__((ext_vector_type(2))) float f32x2;
__device__ __forceinline__ f32x2 line_take(const float* at) {
  const unsigned long long v = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return f32x2{__uint_as_float((unsigned)v), __uint_as_float((unsigned)(v >> 32))};
}
// whether this workgroup is the first of its tile (the same in all threads; lds: an int that nobody else uses)
__device__ __forceinline__ bool line_first(const LineArgs& a, const LineTile& t, int* lds) {
  if (threadIdx.x == 0) *lds = __hip_atomic_fetch_add(a.met + 2 * t.rest, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  const bool first = *lds == 0;
  __syncthreads();
  return first;
}
__device__ __forceinline__ void line_ready(const LineArgs& a, const LineTile& t) {      // behind the first one's last line_give
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's sums are in memory
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(a.met + 2 * t.rest + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void line_await(const LineArgs& a, const LineTile& t) {      // in front of the second one's first line_take
  if (threadIdx.x == 0) {
    while (!__hip_atomic_load(a.met + 2 * t.rest + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) __builtin_amdgcn_s_sleep(1);
    __hip_atomic_store(a.met + 2 * t.rest, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // for the next launch
    __hip_atomic_store(a.met + 2 * t.rest + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
}
__device__ __forceinline__ const bf16_t* line_row(const LineArgs& a, const LineTile& t, int row) {
  const int m = min(t.mbase + row, t.mend - 1);      // rows past the end are computed on a clamped row, never stored
  return a.terms + (size_t)(a.g.a_rows ? a.g.a_rows[m] : m) * a.ldt + (size_t)t.z * 2 * a.g.a_zoff;
}
// weight row of a tile's local column; dual: blocks of 32 columns of the first and the second matrix in turn
template <bool DUAL, int TN>
__device__ __forceinline__ const bf16_t* line_col(const LineArgs& a, const LineTile& t, int local) {
  const int n = DUAL ? t.tn * (TN / 2) + (local >> 6) * 32 + (local & 31) : t.tn * TN + local;
  const void* B = DUAL && (local & 32) ? a.g.B2 : a.g.B;
  return reinterpret_cast<const bf16_t*>(B) + (size_t)t.z * a.g.b_zstride + (size_t)min(n, a.g.N - 1) * a.g.ldb;
}

// Epilogues go through LDS: unrolled over a lane's 64 to 128 accumulators, an epilogue with its choice of activations is more code than the instruction cache holds (2048 rows
// 2048 x 2048: 83 us for a 45 us loop), and a lane's outputs are single columns.  Staged rows of LINE_RS floats (a row's fours stay 16-byte aligned; the two half waves
// of an accumulator write, four rows apart, fall on different banks) are taken four columns at a time by a rolled loop.
constexpr int LINE_RS = 136;
// four outputs of row m from column n on (of one matrix)
template <int DT, int EPI, bool PLAIN>
__device__ __forceinline__ void line_out4(const LineArgs& a, const LineTile& t, int m, int n, const f32x4 v, const f32x4 v2) {
  if (m >= t.mend || n >= a.g.N) return;
  const size_t crow = a.g.c_rows ? (size_t)a.g.c_rows[m] : (size_t)m;
  float* cp = a.g.C + crow * a.g.ldc + (size_t)t.z * a.g.c_zoff + n;
  const bool whole = n + 3 < a.g.N && ((uintptr_t)cp & 15) == 0;
  f32x4 old = {0.f, 0.f, 0.f, 0.f}, o;
  if constexpr (EPI == SG_ADD) {
    if (whole) old = *reinterpret_cast<const f32x4*>(cp);
    else
#pragma unroll
      for (int e = 0; e < 4; e++) if (n + e < a.g.N) old[e] = cp[e];
  }
#pragma unroll
  for (int e = 0; e < 4; e++) o[e] = PLAIN ? v[e] * a.g.scale : n + e < a.g.N ? sg_value<EPI>(a.g, t.z, m, crow, n + e, v[e], v2[e], old[e]) : 0.f;
  if (a.g.Ct) {      // as the next product's lines (N a multiple of 64)
    bf16_t h[4], l[4];
#pragma unroll
    for (int e = 0; e < 4; e++) { split16<DT>(o[e], h[e], l[e]); if (a.g.terms == 1) l[e] = 0; }
    bf16_t* line = a.g.Ct + (crow * (a.g.N >> 5) + (n >> 5)) * 64 + (n & 31);
    *reinterpret_cast<u32x2*>(line) = u32x2{(unsigned int)h[0] | ((unsigned int)h[1] << 16), (unsigned int)h[2] | ((unsigned int)h[3] << 16)};
    *reinterpret_cast<u32x2*>(line + 32) = u32x2{(unsigned int)l[0] | ((unsigned int)l[1] << 16), (unsigned int)l[2] | ((unsigned int)l[3] << 16)};
  } else if (whole) *reinterpret_cast<f32x4*>(cp) = o;
  else
#pragma unroll
    for (int e = 0; e < 4; e++) if (n + e < a.g.N) cp[e] = o[e];
}
// `rows` staged rows from row0 of the tile on: TN staged columns each (dual: blocks of 32 of the two matrices in turn), dealt in fours to `nthr` threads.  sum: a second set of
// staged rows to be added
template <int DT, int EPI, bool DUAL, int TN, bool SUM>
__device__ __forceinline__ void line_epilogue(const LineArgs& a, const LineTile& t, const float* st, const float* sum, int rows, int row0, int n0, int thr, int nthr) {
  constexpr int QUADS = TN / (DUAL ? 8 : 4);      // fours of outputs per row
  auto loop = [&](auto PLAINc, auto Uc) {
    constexpr bool PLAIN = decltype(PLAINc)::value; constexpr int U = decltype(Uc)::value;
#pragma unroll U
    for (int q = thr; q < rows * QUADS; q += nthr) {
      const int row = q / QUADS, c = (q % QUADS) * 4, sc = DUAL ? (c >> 5) * 64 + (c & 31) : c;
      f32x4 v = *reinterpret_cast<const f32x4*>(st + row * LINE_RS + sc), v2 = v;
      if constexpr (SUM) v += *reinterpret_cast<const f32x4*>(sum + row * LINE_RS + sc);
      if constexpr (DUAL) {
        v2 = *reinterpret_cast<const f32x4*>(st + row * LINE_RS + sc + 32);
        if constexpr (SUM) v2 += *reinterpret_cast<const f32x4*>(sum + row * LINE_RS + sc + 32);
      }
      line_out4<DT, EPI, PLAIN>(a, t, t.mbase + row0 + row, n0 + c, v, v2);
    }
  };
  const bool plain = EPI == SG_STORE && !a.g.bias && !a.g.in_w && a.g.act == SG_ACT_NONE && a.g.gate_heads <= 0;
  if (EPI == SG_STORE && plain) loop(std::true_type{}, std::integral_constant<int, 4>{});
  else loop(std::false_type{}, std::integral_constant<int, EPI == SG_ADD || EPI == SG_ROWSCALE ? 4 : 1>{});
}

template <int DT, int EPI, bool DUAL, bool SHARED>
__global__ __launch_bounds__(512) void stack_line256_kernel(const LineArgs a) {
  constexpr int TMN = 256, NSLOT = 5, UNIT = TMN * 64;     // 16-bit elements per unit: 256 rows x 128 bytes
  extern __shared__ __attribute__((aligned(1024))) bf16_t dma_lds[];
  LineTile t;
  if (!line_place<SHARED>(a, TMN, t)) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv >> 1, wn = wv & 1;
  const unsigned lds_base = (unsigned)(size_t)dma_lds;
  f32x16 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

  // DMA map: a unit = 32 pieces of 8 rows x 128 bytes; wave w takes pieces w, w + 8, w + 16, w + 24; chunk c of row r sits in slot c ^ ((r >> 1) & 7)
  const int prow = lane >> 3, pslot = lane & 7;
  const bf16_t *srcA[4], *srcB[4];
#pragma unroll
  for (int p = 0; p < 4; p++) {
    const int row = (wv + 8 * p) * 8 + prow, chunk = pslot ^ ((row >> 1) & 7);
    srcA[p] = line_row(a, t, row) + (size_t)t.k0 * 128 + chunk * 8;
    srcB[p] = line_col<DUAL, TMN>(a, t, row) + (size_t)t.k0 * 64 + chunk * 8;
  }
  const int nblk = t.nk;
  // unit u = 3 b + j: j = 0 the A lines of step 2b, 1 the B lines of block b, 2 the A lines of step 2b + 1 (units past the end reload the last block)
  auto issue = [&](int b, int j, int p) {
    const int bb = min(b, nblk - 1);
    const unsigned dst = lds_base + (unsigned)(((3 * b + j) % NSLOT) * UNIT * 2) + (unsigned)((wv + 8 * p) * 1024);
    if (j == 1) dma_1k(srcB[p] + (size_t)bb * 64, dst);
    else dma_1k(srcA[p] + (size_t)(2 * bb + (j >> 1)) * 64, dst);
  };
  const int swz = ((lane & 31) >> 1) & 7;
  const int arow = (wm * 64 + (lane & 31)) * 64, brow_l = (wn * 128 + (lane & 31)) * 64;
  auto read_frags = [&](int s, int kk, bf16x8* fa, bf16x8* fb) {
    const int b = s >> 1;
    const bf16_t* ua = dma_lds + (size_t)((3 * b + ((s & 1) << 1)) % NSLOT) * UNIT;
    const bf16_t* ub = dma_lds + (size_t)((3 * b + 1) % NSLOT) * UNIT;
    const int ca = kk * 2 + (lane >> 5), cb = (s & 1) * 4 + ca;
#pragma unroll
    for (int j = 0; j < 4; j++) fb[j] = *reinterpret_cast<const bf16x8*>(ub + brow_l + j * 32 * 64 + ((cb ^ swz) << 3));
#pragma unroll
    for (int i = 0; i < 2; i++) {
      fa[2 * i] = *reinterpret_cast<const bf16x8*>(ua + arow + i * 32 * 64 + ((ca ^ swz) << 3));
      fa[2 * i + 1] = *reinterpret_cast<const bf16x8*>(ua + arow + i * 32 * 64 + (((4 + ca) ^ swz) << 3));
    }
  };
  auto mfma_step = [&](const bf16x8* fa, const bf16x8* fb, int b, int j, int p0, int np) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
#pragma unroll
      for (int p = 0; p < 2; p++) {
        const int idx = 2 * g + p, i = idx / 4, jj = idx % 4;
        acc[i][jj] = mfma16<DT>(fa[2 * i + 1], fb[jj], acc[i][jj]);   // small term first
        acc[i][jj] = mfma16<DT>(fa[2 * i], fb[jj], acc[i][jj]);
      }
      if (g < np) issue(b, j, p0 + g);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int u = 0; u < 5; u++)
#pragma unroll
    for (int p = 0; p < 4; p++) issue(u / 3, u % 3, p);
  bf16x8 fa0[4], fb0[4], fa1[4], fb1[4];
  asm volatile("s_waitcnt vmcnt(12)" ::: "memory");          // units 0, 1 landed (this wave's pieces); units 2, 3, 4 may fly
  __builtin_amdgcn_s_barrier();
  read_frags(0, 0, fa0, fb0);
  for (int b = 0; b < nblk; b++) {
    const int s = 2 * b;
    read_frags(s, 1, fa1, fb1);
    __builtin_amdgcn_sched_barrier(0);
    mfma_step(fa0, fb0, b + 1, 1, 0, b > 0 ? 4 : 0);          // unit 3b+4 = B of block b+1 (the prologue issued block 1's)
    asm volatile("s_waitcnt vmcnt(8)\n\ts_waitcnt lgkmcnt(0)" ::: "memory");      // unit 3b+2 landed: behind it only units 3b+3, 3b+4
    __builtin_amdgcn_s_barrier();                               // every wave has read the A lines of step 2b: unit 3b is free
    read_frags(s + 1, 0, fa0, fb0);
    __builtin_amdgcn_sched_barrier(0);
    mfma_step(fa1, fb1, b + 1, 2, 0, 3);                        // unit 3b+5 = A of step 2b+3, pieces 0..2
    read_frags(s + 1, 1, fa1, fb1);
    __builtin_amdgcn_sched_barrier(0);
    mfma_step(fa0, fb0, b + 1, 2, 3, 1);                        // ... piece 3
    asm volatile("s_waitcnt vmcnt(4)\n\ts_waitcnt lgkmcnt(0)" ::: "memory");      // units 3b+3, 3b+4 landed: behind them only unit 3b+5
    __builtin_amdgcn_s_barrier();                               // units 3b+1 (B) and 3b+2 are free
    read_frags(s + 2, 0, fa0, fb0);                             // (after the last block: a harmless read of a reloaded unit)
    __builtin_amdgcn_sched_barrier(0);
    mfma_step(fa1, fb1, b + 2, 0, 0, 4);                        // unit 3b+6 = A of step 2b+4
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();                                 // the ring is free
  if (SHARED && t.rest >= 0) {
    float* at = a.sums + (size_t)t.rest * TMN * TMN + 2 * tid;
    if (line_first(a, t, reinterpret_cast<int*>(dma_lds))) {
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int r = 0; r < 8; r++) line_give(at + ((i * 4 + j) * 8 + r) * 1024, acc[i][j][2 * r], acc[i][j][2 * r + 1]);
      line_ready(a, t);
      return;
    }
    line_await(a, t);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int r = 0; r < 8; r++) {
          const f32x2 v = line_take(at + ((i * 4 + j) * 8 + r) * 1024);
          acc[i][j][2 * r] += v[0];
          acc[i][j][2 * r + 1] += v[1];
        }
  }
  // every wave stages its block, 32 rows at a time, in a slice of its own
  float* st = reinterpret_cast<float*>(dma_lds) + (size_t)wv * 32 * LINE_RS;
#pragma unroll
  for (int i = 0; i < 2; i++) {
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int r = 0; r < 16; r++) st[((r & 3) + 8 * (r >> 2) + 4 * (lane >> 5)) * LINE_RS + j * 32 + (lane & 31)] = acc[i][j][r];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // (the wave reads only what it wrote itself)
    line_epilogue<DT, EPI, DUAL, 128, false>(a, t, st, nullptr, 32, wm * 64 + i * 32, t.tn * (DUAL ? 128 : 256) + wn * (DUAL ? 64 : 128), lane, 64);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

// HALF: the waves are 2 x 2 quadrants x two halves of a stage's k16 steps, not two row halves x four quarters, for chains of up to 32 stages, as in gemm_dma8h_kernel (gemm_dma.h): the sums
// meet in the epilogue, with no exchange in front of it.  Each k16 step has a sum of its own, as there: the same numbers either way.  us quarters / halves: 1999 rows, gate and up of 512
// (K 1024) 21.2 / 20.5, of 2048 45.0 / 43.8, into 1024 columns K 1024 23.1 / 22.4, K 2048 in halved tiles 33.1 / 32.7; 2397 rows, gate and up of 4096 (K 1024) 107.8 / 104.6, into 1024 columns
// K 1024 26.1 / 25.3, K 4096 62.0 / 62.1; 2048 x 2048 x 2048 44.3 / 44.0
template <int DT, int EPI, bool DUAL, bool SHARED, bool HALF>
__global__ __launch_bounds__(512) void stack_line128_kernel(const LineArgs a) {
  constexpr int TMN = 128, NS = 3, T_A = TMN * 64, STAGE = 3 * T_A;      // a stage: A lines of two k32 steps | B lines, 128 rows x 128 bytes each
  extern __shared__ __attribute__((aligned(1024))) bf16_t dma_lds[];
  LineTile t;
  if (!line_place<SHARED>(a, TMN, t)) return;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int NJ = HALF ? 2 : 4, NSTEP = HALF ? 2 : 1;       // blocks of 32 columns, k16 steps of a stage
  const int kq = HALF ? wv >> 2 : wv >> 1, wm = HALF ? (wv >> 1) & 1 : wv & 1, wn = HALF ? wv & 1 : 0;      // half or quarter of every stage's k16 steps, row half, column half
  const unsigned lds_base = (unsigned)(size_t)dma_lds;
  f32x16 acc[NSTEP][2][NJ];                                    // (halves: steps kq and kq + 2)
#pragma unroll
  for (int s = 0; s < NSTEP; s++)
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[s][i][j][r] = 0.f;
  const int prow = lane >> 3, pslot = lane & 7;
  const bf16_t* gsrc[6];
  unsigned ldst[6];
#pragma unroll
  for (int p = 0; p < 2; p++) {
    const int piece = wv + 8 * p, row = piece * 8 + prow, chunk = pslot ^ ((row >> 1) & 7);
    const bf16_t* ar = line_row(a, t, row) + (size_t)t.k0 * 128 + chunk * 8;
    gsrc[3 * p] = ar; gsrc[3 * p + 1] = ar + 64; gsrc[3 * p + 2] = line_col<DUAL, TMN>(a, t, row) + (size_t)t.k0 * 64 + chunk * 8;
    ldst[3 * p] = (unsigned)(piece * 1024); ldst[3 * p + 1] = ldst[3 * p] + (unsigned)(T_A * 2); ldst[3 * p + 2] = ldst[3 * p] + (unsigned)(2 * T_A * 2);
  }
  // stage k: A lines advance by two (128 elements), B lines by one (64)
  auto issue_piece = [&](int q, int k, int stage) { dma_1k(gsrc[q] + (size_t)k * (q % 3 == 2 ? 64 : 128), lds_base + (unsigned)(stage * STAGE * 2) + ldst[q]); };
  const int nk = t.nk;
#pragma unroll
  for (int q = 0; q < 6; q++) issue_piece(q, 0, 0);
  if (nk > 1) {
#pragma unroll
    for (int q = 0; q < 6; q++) issue_piece(q, 1, 1);
  }
  const int swz = ((lane & 31) >> 1) & 7;
  bf16x8 fah[NSTEP][2], fal[NSTEP][2], fb[NSTEP][NJ];
  for (int k = 0; k < nk; k++) {
    if (k + 1 < nk) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");      // stage k landed: only this wave's pieces of stage k + 1 may fly
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    const bool more = k + 2 < nk;
    const int nst = (k + 2) % NS;
    const bf16_t* st = dma_lds + (size_t)(k % NS) * STAGE;
    const bf16_t* tB = st + 2 * T_A;
#pragma unroll
    for (int s = 0; s < NSTEP; s++) {
      const bf16_t* tA = st + (HALF ? s : kq >> 1) * T_A;
      const int ca = (kq & 1) * 2 + (lane >> 5), cb = (kq + 2 * s) * 2 + (lane >> 5);
#pragma unroll
      for (int j = 0; j < NJ; j++) fb[s][j] = *reinterpret_cast<const bf16x8*>(tB + (wn * 64 + j * 32 + (lane & 31)) * 64 + ((cb ^ swz) << 3));
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const bf16_t* row = tA + (wm * 64 + i * 32 + (lane & 31)) * 64;
        fah[s][i] = *reinterpret_cast<const bf16x8*>(row + ((ca ^ swz) << 3));
        fal[s][i] = *reinterpret_cast<const bf16x8*>(row + (((4 + ca) ^ swz) << 3));
      }
    }
#pragma unroll
    for (int s = 0; s < NSTEP; s++)
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) {
          acc[s][i][j] = mfma16<DT>(fal[s][i], fb[s][j], acc[s][i][j]);   // small term first
          acc[s][i][j] = mfma16<DT>(fah[s][i], fb[s][j], acc[s][i][j]);
          const int q = (s * 2 + i) * NJ + j;
          if (more && q < 6) issue_piece(q, k + 2, nst);
        }
  }
  // (q0 + q2) + (q1 + q3).  Halves: q0 + q2 and q1 + q3 lie in one wave, are staged as rows and added by the epilogue.  Quarters: 2, 3 -> LDS -> added by 0, 1 (same row half), whose
  // sums are staged so.  All waves take part in the epilogue
  __builtin_amdgcn_s_barrier();
  float* red = reinterpret_cast<float*>(dma_lds);
  if constexpr (HALF) {
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[0][i][j][r] += acc[1][i][j][r];
  } else {
    if (kq >= 2) {
      float* dst = red + (size_t)(wv - 4) * 8 * 16 * 64;
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) dst[((i * 4 + j) * 16 + r) * 64 + lane] = acc[0][i][j][r];
    }
    __syncthreads();
    if (kq < 2) {
      const float* src = red + (size_t)wv * 8 * 16 * 64;
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int r = 0; r < 16; r++) acc[0][i][j][r] += src[((i * 4 + j) * 16 + r) * 64 + lane];
    }
    __syncthreads();
  }
  if (kq < 2) {
    float* dst = red + (size_t)kq * TMN * LINE_RS;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) dst[(wm * 64 + i * 32 + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5)) * LINE_RS + wn * 64 + j * 32 + (lane & 31)] = acc[0][i][j][r];
  }
  __syncthreads();
  if (SHARED && t.rest >= 0) {
    float* at = a.sums + (size_t)t.rest * TMN * TMN + 2 * tid;
    auto cell = [&](int q) { return reinterpret_cast<f32x4*>(red + (size_t)(q * 16 + (tid >> 5)) * LINE_RS + 4 * (tid & 31)); };      // a thread's four columns of eight rows
    if (line_first(a, t, reinterpret_cast<int*>(red + (size_t)2 * TMN * LINE_RS))) {
#pragma unroll
      for (int q = 0; q < 8; q++) {
        const f32x4 v = *cell(q) + cell(q)[TMN * LINE_RS / 4];
        line_give(at + (2 * q) * 1024, v[0], v[1]);
        line_give(at + (2 * q + 1) * 1024, v[2], v[3]);
      }
      line_ready(a, t);
      return;
    }
    line_await(a, t);
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const f32x2 u = line_take(at + (2 * q) * 1024), v = line_take(at + (2 * q + 1) * 1024);
      *cell(q) = (*cell(q) + cell(q)[TMN * LINE_RS / 4]) + f32x4{u[0], u[1], v[0], v[1]};      // (the same whichever half is second)
      cell(q)[TMN * LINE_RS / 4] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();
  }
  line_epilogue<DT, EPI, DUAL, TMN, true>(a, t, red, red + (size_t)TMN * LINE_RS, TMN, 0, t.tn * (DUAL ? 64 : 128), tid, 512);
}

}  // namespace tgx
