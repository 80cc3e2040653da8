// stack_gemm.h — the matrix products of layered models: C = epilogue(A · Bᵀ) with fp32 activations A [M][K] and stored weights B [N][K].
//   16-bit storage: v_mfma_f32_32x32x16 on the activation's two 16-bit terms (x = hi + lo, 16 significant bits) — or its rounded first term alone
//   (option act.round16) — against the stored weight, fp32 accumulation; fp32 storage: v_mfma_f32_32x32x2_f32, nothing rounded.
// One kernel serves plain, batched and grouped products:
//   batched (blockIdx.z = head):   B advances by b_zstride, the A / C columns by a_zoff / c_zoff per z — per-head products on slices of wide rows
//   grouped (experts):             blockIdx.y walks a tile list (expert, first row) built on the device (moe_plan_kernel); rows are gathered through
//                                  a_rows and scattered through c_rows
//   dual:                          two weight matrices against the same activation tile (an expert's gate and up projections), combined in the epilogue
// Workgroup = 4 waves as 2 x 2, each WT x WT tiles of 32 x 32: 64 WT x 64 WT outputs per workgroup, K in steps of 64 (32 for fp32 storage) staged through LDS with the
// next step's global loads in flight under the MFMAs.  Any M, N, K: rows, columns and the K tail are masked; shapes that break the 16-byte
// alignment of the vector loads take element loads (VEC = false).
#pragma once
#include "prefill.h"

namespace tgx {

enum { SG_ACT_NONE = 0, SG_ACT_TANH = 1, SG_ACT_DECAY = 2, SG_ACT_GELU = 3, SG_ACT_SOFTPLUS = 4, SG_ACT_RELU2 = 5, SG_ACT_HEAD_DECAY = 6, SG_ACT_GELU_TANH = 7 };
enum { SG_STORE = 0, SG_ADD = 1, SG_GATE = 2, SG_EXPERT_ACT = 3, SG_ROWSCALE = 4, SG_SILU_MUL = 5 };
constexpr int ROWS_MAX_PAIRS = 128;      // stack_rows.h: pairs whose choices a workgroup reads
constexpr bool sg_dual(int epi) { return epi == SG_EXPERT_ACT || epi == SG_SILU_MUL; }
struct StackGemmArgs {
  const float* A; long long lda; int a_zoff;
  const int* a_rows;
  const void* B; const void* B2; long long ldb; long long b_zstride;
  float* C; long long ldc; int c_zoff;
  const int* c_rows;
  const int* z_off; const int* tile_z; const int* tile_m0; const int* n_tiles;      // grouped
  int M, N, K;
  float scale;                 // SG_STORE: C = act(acc * scale + bias); SG_ADD: C += acc * scale
  int act;                     // SG_STORE: SG_ACT_NONE, SG_ACT_TANH, SG_ACT_DECAY = exp(-exp(v)) (a decay in (0, 1) from a log-log pre-activation),
                               //           SG_ACT_GELU = v (1 + erf(v / sqrt 2)) / 2, SG_ACT_SOFTPLUS = ln(1 + e^v), SG_ACT_RELU2 = max(v, 0)^2, or SG_ACT_HEAD_DECAY =
                               //           exp(-exp(a_log[n / head_cols]) ln(1 + e^v)) (a decay per channel whose rate has a factor per head)
                               // SG_SILU_MUL: SG_ACT_GELU_TANH takes the tanh form of gelu instead of silu
  const float* a_log; int head_cols;
  const float* in_w; const int* in_rows;         // SG_STORE: row m's product is first multiplied by in_w[in_rows[m]] (in_rows nullptr: in_w[m]; a router weight on its expert's input; in_w nullptr: none)
  const float* bias;           // SG_STORE: [N] per z (column z * c_zoff + n), nullptr: none
  int gate_col0, gate_heads;   // SG_STORE: columns [gate_col0, + gate_heads) leave as log input gates cap tanh(v / cap), the next gate_heads columns as log forget gates
  float gate_cap;              //           logsigmoid(cap tanh(v / cap)) (the two gate rows of a matrix-memory layer's input product); gate_heads 0: none
  float limit;                 // SG_EXPERT_ACT
  const float* G; long long ldg; int g_col0;     // SG_GATE: C = acc * sigmoid(G[row][g_col0 + z * c_zoff + n]), or with g_per_z
  int g_per_z;                                   //          one gate per batch member z (a head): sigmoid(G[row][g_col0 + z])
  const float* rw;             // SG_ROWSCALE: C = acc * rw[c row]
  int terms;                   // 16-bit storage: 2 = hi + lo, 1 = hi only
  // stack_line.h: the activations, or the outputs, as lines of two 16-bit terms [row][K / 32][hi 32 | lo 32] in the place of A, or of C (nullptr: fp32)
  const unsigned short* At; unsigned short* Ct;
  int a_count;                 // gathered products (a_rows): rows of A
  // one- and two-row products (NORM): A's rows are normed on the way, A / sqrt(mean(A^2) + norm_eps) * (norm_offset + norm_w)
  const float* norm_w; float norm_offset, norm_eps;
  // stack_rows.h: the choices of a step's pairs (an expert each; those from `experts` on have no product); pair p reads row p / pairs_per_row of A and writes row p of C
  const int* sel; int n_pairs, experts, pairs_per_row, tokens;
};

// an expert's activation: g = min(gate, limit), u = clamp(up, -limit, limit); g * sigmoid(1.702 g) * (u + 1)
__device__ __forceinline__ float expert_act(float gate, float up, float limit) {
  const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
  return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
}
// log-space gates of a matrix-memory layer: soft cap, and log sigmoid in the form that loses nothing for large |z|
__device__ __forceinline__ float soft_cap(float z, float cap) { return cap * tanhf(z / cap); }
__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ float store_value(const StackGemmArgs& a, float v, size_t bias_at, int n) {
  float o = a.bias ? fmaf(v, a.scale, a.bias[bias_at]) : v * a.scale;
  if (a.gate_heads > 0 && n >= a.gate_col0) { o = soft_cap(o, a.gate_cap); if (n >= a.gate_col0 + a.gate_heads) o = log_sigmoid(o); }
  if (a.act == SG_ACT_TANH) o = tanhf(o);
  else if (a.act == SG_ACT_DECAY) o = expf(-expf(o));
  else if (a.act == SG_ACT_SOFTPLUS) o = o > 20.f ? o : log1pf(expf(o));
  else if (a.act == SG_ACT_RELU2) { o = fmaxf(o, 0.f); o *= o; }
  else if (a.act == SG_ACT_HEAD_DECAY) o = expf(-expf(a.a_log[n / a.head_cols]) * (o > 20.f ? o : log1pf(expf(o))));
  else if (a.act == SG_ACT_GELU) o = 0.5f * o * (1.0f + erff(o * 0.70710678118654752f));
  return o;
}
// the plain gated expert: silu(gate) * up
__device__ __forceinline__ float silu_mul(float gate, float up) { return gate / (1.0f + expf(-gate)) * up; }
__device__ __forceinline__ float gelu_tanh(float z) { return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * fmaf(0.044715f * z * z, z, z))); }
// the product of a gated feed-forward's two halves: silu or (act SG_ACT_GELU_TANH) the tanh gelu of the gate
__device__ __forceinline__ float gate_mul(const StackGemmArgs& a, float gate, float up) { return a.act == SG_ACT_GELU_TANH ? gelu_tanh(gate) * up : silu_mul(gate, up); }

// the epilogue on the accumulated sum v (dual products: v of the first matrix, v2 of the second) of grouped / batched row m, row crow and column n of C; old: what C holds (SG_ADD)
template <int EPI>
__device__ __forceinline__ float sg_value(const StackGemmArgs& a, int z, int m, size_t crow, int n, float v, float v2, float old) {
  if constexpr (EPI == SG_STORE) return store_value(a, a.in_w ? v * a.in_w[a.in_rows ? a.in_rows[m] : m] : v, (size_t)z * a.c_zoff + n, n);
  else if constexpr (EPI == SG_ADD) return fmaf(v, a.scale, old);
  else if constexpr (EPI == SG_GATE) return v / (1.0f + expf(-a.G[crow * a.ldg + a.g_col0 + (a.g_per_z ? (size_t)z : (size_t)z * a.c_zoff + n)]));
  else if constexpr (EPI == SG_EXPERT_ACT) return expert_act(v, v2, a.limit);
  else if constexpr (EPI == SG_SILU_MUL) return gate_mul(a, v, v2);
  else return v * a.rw[crow];
}
// one output of a product
template <int EPI>
__device__ __forceinline__ void sg_finish(const StackGemmArgs& a, int z, int m, int n, float v, float v2) {
  const size_t crow = a.c_rows ? (size_t)a.c_rows[m] : (size_t)m;
  float* cp = a.C + crow * a.ldc + (size_t)z * a.c_zoff + n;
  *cp = sg_value<EPI>(a, z, m, crow, n, v, v2, EPI == SG_ADD ? *cp : 0.f);
}

template <int DT, int EPI, bool DUAL, int WT, bool VEC>
__global__ __launch_bounds__(256) void stack_gemm_kernel(const StackGemmArgs a) {
  constexpr bool F32 = DT == DT_F32;
  constexpr int BM = 64 * WT, BN = 64 * WT, BK = F32 ? 32 : 64;      // 16-bit tiles take 64 k per step: half the barriers, twice the bytes in flight
  constexpr int ACH = BK / 4, BCH = F32 ? BK / 4 : BK / 8;            // 16-byte chunks per staged row
  constexpr int LDK = BK + 8;                       // 16-bit tiles: row-major, k contiguous, 16 bytes of padding
  constexpr int LDA = BM + 1, LDB = BN + 1;         // fp32 tiles: k-major
  constexpr int NB = DUAL ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16_t* sAh = reinterpret_cast<bf16_t*>(smem);
  bf16_t* sAl = sAh + BM * LDK;
  bf16_t* sB = sAl + BM * LDK;                      // [NB][BN][LDK]
  float* fA = reinterpret_cast<float*>(smem);       // [BK][LDA]
  float* fB = fA + BK * LDA;                        // [NB][BK][LDB]

  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, wm = wv >> 1, wn = wv & 1;
  int z, mbase, mend;
  if (a.z_off) {
    if ((int)blockIdx.y >= *a.n_tiles) return;
    z = a.tile_z[blockIdx.y]; mbase = a.tile_m0[blockIdx.y]; mend = a.z_off[z + 1];
  } else { z = blockIdx.z; mbase = blockIdx.y * BM; mend = a.M; }
  const int n0 = blockIdx.x * BN;
  const float* Ab = a.A + (size_t)z * a.a_zoff;
  const elem_t<DT>* Bz[NB];
  Bz[0] = reinterpret_cast<const elem_t<DT>*>(a.B) + (size_t)z * a.b_zstride;
  if constexpr (DUAL) Bz[1] = reinterpret_cast<const elem_t<DT>*>(a.B2) + (size_t)z * a.b_zstride;

  f32x16 acc[NB][WT][WT];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
      for (int j = 0; j < WT; j++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[b][i][j][r] = 0.f;

  // ---- staging maps.  A: chunks of 4 k (fp32) -> chunk c: row c / ACH, k 4 (c % ACH).  B: 16-bit chunks of 8 k -> row c / BCH, k 8 (c % BCH); fp32 as A.
  constexpr int AI = BM * (BK / 4) / 256;
  constexpr int BI = F32 ? BN * (BK / 4) / 256 : BN * (BK / 8) / 256;
  f32x4 ra[AI];
  f32x4 rbf[F32 ? NB * BI : 1];
  u32x4 rbh[F32 ? 1 : NB * BI];
  size_t arow[AI];
#pragma unroll
  for (int i = 0; i < AI; i++) {
    const int m = mbase + (tid + 256 * i) / ACH;
    const int mc = min(m, mend - 1);
    arow[i] = (size_t)(a.a_rows ? a.a_rows[mc] : mc) * a.lda;
  }
  auto load_tiles = [&](int k0) {
#pragma unroll
    for (int i = 0; i < AI; i++) {
      const int k = k0 + 4 * ((tid + 256 * i) % ACH);
      const float* p = Ab + arow[i] + k;
      if (VEC) ra[i] = k < a.K ? *reinterpret_cast<const f32x4*>(p) : f32x4{0.f, 0.f, 0.f, 0.f};
      else
#pragma unroll
        for (int e = 0; e < 4; e++) ra[i][e] = k + e < a.K ? p[e] : 0.f;
    }
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int i = 0; i < BI; i++) {
        const int c = tid + 256 * i;
        if constexpr (F32) {
          const int n = min(n0 + c / BCH, a.N - 1), k = k0 + 4 * (c % BCH);
          const float* p = reinterpret_cast<const float*>(Bz[b]) + (size_t)n * a.ldb + k;
          if (VEC) rbf[b * BI + i] = k < a.K ? *reinterpret_cast<const f32x4*>(p) : f32x4{0.f, 0.f, 0.f, 0.f};
          else
#pragma unroll
            for (int e = 0; e < 4; e++) rbf[b * BI + i][e] = k + e < a.K ? p[e] : 0.f;
        } else {
          const int n = min(n0 + c / BCH, a.N - 1), k = k0 + 8 * (c % BCH);
          const bf16_t* p = reinterpret_cast<const bf16_t*>(Bz[b]) + (size_t)n * a.ldb + k;
          if (VEC) rbh[b * BI + i] = k < a.K ? *reinterpret_cast<const u32x4*>(p) : u32x4{0u, 0u, 0u, 0u};
          else {
            u32x4 v = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int e = 0; e < 8; e++) if (k + e < a.K) v[e >> 1] |= (unsigned int)p[e] << (16 * (e & 1));
            rbh[b * BI + i] = v;
          }
        }
      }
  };
  auto store_tiles = [&]() {
#pragma unroll
    for (int i = 0; i < AI; i++) {
      const int c = tid + 256 * i, row = c / ACH, kc = c % ACH;
      if constexpr (F32) {
#pragma unroll
        for (int e = 0; e < 4; e++) fA[(4 * kc + e) * LDA + row] = ra[i][e];
      } else {
        bf16_t h[4], l[4];
#pragma unroll
        for (int e = 0; e < 4; e++) split16<DT>(ra[i][e], h[e], l[e]);
        *reinterpret_cast<u32x2*>(sAh + row * LDK + 4 * kc) = u32x2{(unsigned int)h[0] | ((unsigned int)h[1] << 16), (unsigned int)h[2] | ((unsigned int)h[3] << 16)};
        *reinterpret_cast<u32x2*>(sAl + row * LDK + 4 * kc) = u32x2{(unsigned int)l[0] | ((unsigned int)l[1] << 16), (unsigned int)l[2] | ((unsigned int)l[3] << 16)};
      }
    }
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int i = 0; i < BI; i++) {
        const int c = tid + 256 * i;
        if constexpr (F32) {
          const int row = c / BCH, kc = c % BCH;
#pragma unroll
          for (int e = 0; e < 4; e++) fB[(b * BK + 4 * kc + e) * LDB + row] = rbf[b * BI + i][e];
        } else {
          const int row = c / BCH, kc = c % BCH;
          *reinterpret_cast<u32x4*>(sB + ((size_t)b * BN + row) * LDK + 8 * kc) = rbh[b * BI + i];
        }
      }
  };

  load_tiles(0);
  for (int k0 = 0; k0 < a.K; k0 += BK) {
    __syncthreads();
    store_tiles();
    __syncthreads();
    if (k0 + BK < a.K) load_tiles(k0 + BK);
    if constexpr (F32) {
#pragma unroll
      for (int kk = 0; kk < BK / 2; kk++) {
        const int krow = 2 * kk + (lane >> 5);
        float fa[WT], fb[NB][WT];
#pragma unroll
        for (int i = 0; i < WT; i++) fa[i] = fA[krow * LDA + wm * (32 * WT) + i * 32 + (lane & 31)];
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int j = 0; j < WT; j++) fb[b][j] = fB[(b * BK + krow) * LDB + wn * (32 * WT) + j * 32 + (lane & 31)];
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int i = 0; i < WT; i++)
#pragma unroll
            for (int j = 0; j < WT; j++) acc[b][i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[b][j], acc[b][i][j], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < BK / 16; kk++) {
        const int kof = 16 * kk + 8 * (lane >> 5);
        bf16x8 ah[WT], al[WT], bb[NB][WT];
#pragma unroll
        for (int i = 0; i < WT; i++) {
          const int row = wm * (32 * WT) + i * 32 + (lane & 31);
          ah[i] = *reinterpret_cast<const bf16x8*>(sAh + row * LDK + kof);
          al[i] = *reinterpret_cast<const bf16x8*>(sAl + row * LDK + kof);
        }
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int j = 0; j < WT; j++) bb[b][j] = *reinterpret_cast<const bf16x8*>(sB + ((size_t)b * BN + wn * (32 * WT) + j * 32 + (lane & 31)) * LDK + kof);
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
          for (int i = 0; i < WT; i++)
#pragma unroll
            for (int j = 0; j < WT; j++) {
              acc[b][i][j] = mfma16<DT>(ah[i], bb[b][j], acc[b][i][j]);
              if (a.terms > 1) acc[b][i][j] = mfma16<DT>(al[i], bb[b][j], acc[b][i][j]);
            }
      }
    }
  }

  // ---- epilogue.  C / D layout of the 32 x 32 product: column = lane & 31, row = (r & 3) + 8 (r >> 2) + 4 (lane >> 5)
#pragma unroll
  for (int i = 0; i < WT; i++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int m = mbase + wm * (32 * WT) + i * 32 + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5);
      if (m >= mend) continue;
#pragma unroll
      for (int j = 0; j < WT; j++) {
        const int n = n0 + wn * (32 * WT) + j * 32 + (lane & 31);
        if (n < a.N) sg_finish<EPI>(a, z, m, n, acc[0][i][j][r], acc[NB - 1][i][j][r]);
      }
    }
}

template <int DT, bool DUAL, int WT>
constexpr size_t stack_gemm_lds() {
  constexpr int BM = 64 * WT, BN = 64 * WT, BK = DT == DT_F32 ? 32 : 64, NB = DUAL ? 2 : 1;
  return DT == DT_F32 ? (size_t)(BK * (BM + 1) + NB * BK * (BN + 1)) * 4 : (size_t)(2 * BM + NB * BN) * (BK + 8) * 2;
}

}  // namespace tgx

namespace tgx {

constexpr int STACK_GEMV_COLS = 2;      // output columns per wave

// ---- the same products for ONE or TWO rows (decode steps): a weight-streaming kernel.  One wave per pair of output columns: every lane takes 8 weights of each
// column per pass (one 16-byte load for the 16-bit dtypes) against the 8 activations of up to MR rows, fp32 FMA chains, one cross-lane sum per (row, column)
// at the end.  KSPLIT: the four waves divide the slices of one pair of columns (their sums meet in LDS): four times the workgroups.  Same argument block, batching (blockIdx.z) and epilogues as stack_gemm_kernel; the activations
// enter in fp32 (rounded to the storage dtype first under option act.round16).  Needs the vector-load alignment (K a multiple of 8).
template <int DT, int EPI, bool DUAL, int MR, bool KSPLIT = false>
__device__ __forceinline__ void stack_gemv_body(const StackGemmArgs& a, int bx, int by, int z) {
  constexpr int NC = STACK_GEMV_COLS, NB = DUAL ? 2 : 1;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int mbase = by * MR, mend = min(a.M, mbase + MR);
  const int n0 = (KSPLIT ? bx : bx * (int)(blockDim.x >> 6) + wv) * NC;
  if (n0 >= a.N) return;
  const float* Ab = a.A + (size_t)z * a.a_zoff;
  const float* arow[MR];
#pragma unroll
  for (int r = 0; r < MR; r++) { const int mc = min(mbase + r, mend - 1); arow[r] = Ab + (size_t)(a.a_rows ? a.a_rows[mc] : mc) * a.lda; }
  const elem_t<DT>* wrow[NB][NC];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int j = 0; j < NC; j++)
      wrow[b][j] = reinterpret_cast<const elem_t<DT>*>(b ? a.B2 : a.B) + (size_t)z * a.b_zstride + (size_t)min(n0 + j, a.N - 1) * a.ldb;
  float acc[NB][NC][MR];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int j = 0; j < NC; j++)
#pragma unroll
      for (int r = 0; r < MR; r++) acc[b][j][r] = 0.f;
  const int round16 = a.terms == 1;
  const int nsl = a.K >> 3;                               // 8-element slices of a row
  for (int s0 = KSPLIT ? 64 * wv + lane : lane; s0 < nsl; s0 += KSPLIT ? 512 : 128) {              // two slices per lane and pass: twice the loads in flight
    const int s1 = s0 + (KSPLIT ? 256 : 64);
    const bool two = s1 < nsl;
    Slice8<DT> w0[NB][NC], w1[NB][NC];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int j = 0; j < NC; j++) { w0[b][j] = load_slice_nt<DT>(wrow[b][j], (size_t)s0); w1[b][j] = load_slice_nt<DT>(wrow[b][j], (size_t)(two ? s1 : s0)); }
#pragma unroll
    for (int r = 0; r < MR; r++) {
      const f32x4* xp = reinterpret_cast<const f32x4*>(arow[r]);
      f32x4 xa = xp[2 * s0], xb = xp[2 * s0 + 1], ya = xp[2 * (two ? s1 : s0)], yb = xp[2 * (two ? s1 : s0) + 1];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        xa[i] = round_storage_if<DT>(xa[i], round16); xb[i] = round_storage_if<DT>(xb[i], round16);
        ya[i] = two ? round_storage_if<DT>(ya[i], round16) : 0.f; yb[i] = two ? round_storage_if<DT>(yb[i], round16) : 0.f;
      }
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int j = 0; j < NC; j++) { acc[b][j][r] = dot8<DT>(acc[b][j][r], w0[b][j], xa, xb); acc[b][j][r] = dot8<DT>(acc[b][j][r], w1[b][j], ya, yb); }
    }
  }
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int j = 0; j < NC; j++)
#pragma unroll
      for (int r = 0; r < MR; r++) acc[b][j][r] = wave_sum(acc[b][j][r]);
  if constexpr (KSPLIT) {
    __shared__ float s_part[4][NB * NC * MR];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int j = 0; j < NC; j++)
#pragma unroll
        for (int r = 0; r < MR; r++) if (lane == 0) s_part[wv][(b * NC + j) * MR + r] = acc[b][j][r];
    __syncthreads();
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int j = 0; j < NC; j++)
#pragma unroll
        for (int r = 0; r < MR; r++) { const int at = (b * NC + j) * MR + r; acc[b][j][r] = s_part[0][at] + s_part[1][at] + s_part[2][at] + s_part[3][at]; }
    if (wv) return;
  }
  // one output a lane, so that the epilogues' loads (bias, gate, the stream itself) are one round trip and not one after the other
  float v = acc[0][0][0], v2 = acc[NB - 1][0][0];
#pragma unroll
  for (int r = 0; r < MR; r++)
#pragma unroll
    for (int j = 0; j < NC; j++)
      if (lane == r * NC + j) { v = acc[0][j][r]; v2 = acc[NB - 1][j][r]; }
  const int m = mbase + lane / NC, n = n0 + lane % NC;
  if (lane < MR * NC && m < mend && n < a.N) sg_finish<EPI>(a, z, m, n, v, v2);
}
// ---- the same where the rows are a stream in front of its RMS norm: rows / sqrt(mean(row^2) + norm_eps) * (norm_offset + norm_w).  A workgroup's first weights are on their way before
// its threads read the rows, times the norm's weights, into LDS and sum their squares; the norm's factor multiplies the products at the end.  One launch less (2.3 to 3.6 us), and a row
// is read once a workgroup instead of once a wave: the output product of 32000 x 1024 14.7 + 2.3 -> 12.8 us (5.1 TB/s), of 32000 x 2048 24.2 + 3.6 -> 22.5 (5.8).  Up to GEMV_NORM_MAX
// channels.
constexpr int GEMV_NORM_MAX = 4096;
template <int DT, int EPI, bool DUAL, int MR, int NW>
__device__ __forceinline__ void stack_gemv_norm_body(const StackGemmArgs& a, int bx) {
  constexpr int NC = STACK_GEMV_COLS, NB = DUAL ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) float s_row[];      // [MR][K]
  __shared__ float s_ss[MR][NW];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, n0 = (bx * NW + wv) * NC, nsl = a.K >> 3;
  const elem_t<DT>* wrow[NB][NC];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int j = 0; j < NC; j++) wrow[b][j] = reinterpret_cast<const elem_t<DT>*>(b ? a.B2 : a.B) + (size_t)min(n0 + j, a.N - 1) * a.ldb;
  Slice8<DT> w0[NB][NC], w1[NB][NC];
  auto load = [&](int s0) {      // two slices per lane (past the end: the last again, dropped)
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int j = 0; j < NC; j++) { w0[b][j] = load_slice_nt<DT>(wrow[b][j], (size_t)min(s0, nsl - 1)); w1[b][j] = load_slice_nt<DT>(wrow[b][j], (size_t)min(s0 + 64, nsl - 1)); }
  };
  load(lane);
#pragma unroll
  for (int r = 0; r < MR; r++) {
    const int mc = min(r, a.M - 1);
    const float* row = a.A + (size_t)(a.a_rows ? a.a_rows[mc] : mc) * a.lda;
    float ss = 0.f;
    for (int c = 4 * threadIdx.x; c < a.K; c += 256 * NW) {
      f32x4 x = *reinterpret_cast<const f32x4*>(row + c);
      const f32x4 g = *reinterpret_cast<const f32x4*>(a.norm_w + c);
#pragma unroll
      for (int i = 0; i < 4; i++) { ss = fmaf(x[i], x[i], ss); x[i] *= a.norm_offset + g[i]; }
      *reinterpret_cast<f32x4*>(s_row + (size_t)r * a.K + c) = x;
    }
    ss = group_sum<64>(ss);
    if (lane == 0) s_ss[r][wv] = ss;
  }
  __syncthreads();
  if (n0 >= a.N) return;
  float acc[NB][NC][MR];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int j = 0; j < NC; j++)
#pragma unroll
      for (int r = 0; r < MR; r++) acc[b][j][r] = 0.f;
  for (int s0 = lane; s0 - lane < nsl; s0 += 128) {
    if (s0 >= 128) load(s0);
    const int s1 = s0 + 64;
#pragma unroll
    for (int r = 0; r < MR; r++) {
      const f32x4* xp = reinterpret_cast<const f32x4*>(s_row + (size_t)r * a.K);
      const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
      const int c0 = min(s0, nsl - 1), c1 = min(s1, nsl - 1);
      f32x4 xa = xp[2 * c0], xb = xp[2 * c0 + 1], ya = xp[2 * c1], yb = xp[2 * c1 + 1];
      if (s0 >= nsl) xa = xb = zero;
      if (s1 >= nsl) ya = yb = zero;
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int j = 0; j < NC; j++) { acc[b][j][r] = dot8<DT>(acc[b][j][r], w0[b][j], xa, xb); acc[b][j][r] = dot8<DT>(acc[b][j][r], w1[b][j], ya, yb); }
    }
  }
#pragma unroll
  for (int r = 0; r < MR; r++) {
    float ss = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) ss += s_ss[r][w];
    const float f = 1.0f / sqrtf(ss / (float)a.K + a.norm_eps);
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int j = 0; j < NC; j++) acc[b][j][r] = wave_sum(acc[b][j][r]) * f;
  }
  float v = acc[0][0][0], v2 = acc[NB - 1][0][0];
#pragma unroll
  for (int r = 0; r < MR; r++)
#pragma unroll
    for (int j = 0; j < NC; j++)
      if (lane == r * NC + j) { v = acc[0][j][r]; v2 = acc[NB - 1][j][r]; }
  const int m = lane / NC, n = n0 + lane % NC;
  if (lane < MR * NC && m < a.M && n < a.N) sg_finish<EPI>(a, 0, m, n, v, v2);
}
// a plain product on rows in front of their norm (a model's last)
template <int DT, int MR>
__global__ __launch_bounds__(256) void stack_gemv_norm_kernel(const StackGemmArgs a) { stack_gemv_norm_body<DT, SG_STORE, false, MR, 4>(a, blockIdx.x); }
template <int DT, int EPI, bool DUAL, int MR, bool KSPLIT>
__global__ __launch_bounds__(256) void stack_gemv_kernel(const StackGemmArgs a) { stack_gemv_body<DT, EPI, DUAL, MR, KSPLIT>(a, blockIdx.x, blockIdx.y, blockIdx.z); }

// ---- a layer whose mixer and feed-forward read the same input and add to the same stream.  A decode step is bound by its launches (1024 x 1024 streams 2 MB in 0.4 us and
// takes 2.6), so the products that stand at the same place of the two chains share one:
//   stack_gemv_group_kernel   the mixer's input product (batched by z0), a second plain product of the mixer's (M = 0: none) and the feed-forward's gate and up
//   stack_gemv_sum_kernel     x += sum_s A_s W_s^T scale_s over the outputs of the mixer's parts and of the feed-forward, added in that order
// Grid: the workgroups of the group's products one after the other; (N / 2) for the sum.  Eight layers of 1024 channels, one stream: 89 launches a step become 62, a step
// 360 -> 283 us.
struct StackGemvGroup { StackGemmArgs p0, p1, up; int z0, blocks0, blocks1; };      // blocks0: per member of the batch
// NORM: the rows are the stream in front of the layer's norm: 1 for the feed-forward, 2 for the mixer's first product as well.  NW: waves of a workgroup; with the norm eight up to
// GEMV_GROUP_WIDE channels, whose weights are all on their way before the rows have been read, four beyond.  One row, the group of a wkv and of an attention layer, eight / four waves, us: 512
// channels 9.2 / 9.4, 1024 11.3 / 12.2, 1280 16.8 / 17.7, 1536 20.6 / 19.7, 2048 31 / 25, 3072 34.6 both; two rows are within 6 % of each other at every width.  With the
// norms in launches of their own 1024 10.9 + 5.2, 1536 20.4 + 5.2, 2048 26.5 + 5.1.
constexpr int GEMV_GROUP_WIDE = 1024;
template <int DT, int MR, int NORM, int NW>
__global__ __launch_bounds__(64 * NW) void stack_gemv_group_kernel(const StackGemvGroup g) {
  int b = blockIdx.x;
  if (b < g.blocks0 * g.z0) {
    if constexpr (NORM == 2) stack_gemv_norm_body<DT, SG_STORE, false, MR, NW>(g.p0, b);
    else stack_gemv_body<DT, SG_STORE, false, MR>(g.p0, b % g.blocks0, 0, b / g.blocks0);
    return;
  }
  b -= g.blocks0 * g.z0;
  if (b < g.blocks1) { stack_gemv_body<DT, SG_STORE, false, MR>(g.p1, b, 0, 0); return; }
  if constexpr (NORM != 0) stack_gemv_norm_body<DT, SG_SILU_MUL, true, MR, NW>(g.up, b - g.blocks1);
  else stack_gemv_body<DT, SG_SILU_MUL, true, MR>(g.up, b - g.blocks1, 0, 0);
}
// The four waves of a workgroup divide the slices of all sources of two columns between them, two in flight per lane and pass: W = 1024 would otherwise leave half of the
// compute units without a wave and give the others five round trips.
constexpr int GEMV_SUM_MAX = 3;
struct StackGemvSum { StackGemmArgs p[GEMV_SUM_MAX]; };
template <int DT, int NS, int MR>
__global__ __launch_bounds__(256) void stack_gemv_sum_kernel(const StackGemvSum g) {
  constexpr int NC = STACK_GEMV_COLS;
  __shared__ float s_part[4][NS * NC * MR];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, n0 = blockIdx.x * NC, N = g.p[0].N, M = g.p[0].M;
  float acc[NS][NC][MR];
#pragma unroll
  for (int s = 0; s < NS; s++) {
    const StackGemmArgs& a = g.p[s];
#pragma unroll
    for (int j = 0; j < NC; j++)
#pragma unroll
      for (int r = 0; r < MR; r++) acc[s][j][r] = 0.f;
    const elem_t<DT>* wrow[NC];
#pragma unroll
    for (int j = 0; j < NC; j++) wrow[j] = reinterpret_cast<const elem_t<DT>*>(a.B) + (size_t)min(n0 + j, N - 1) * a.ldb;
    const int nsl = a.K >> 3;
    for (int s0 = 64 * wv + lane; s0 < nsl; s0 += 512) {
      const int s1 = s0 + 256;
      const bool two = s1 < nsl;
      Slice8<DT> w0[NC], w1[NC];
#pragma unroll
      for (int j = 0; j < NC; j++) { w0[j] = load_slice_nt<DT>(wrow[j], (size_t)s0); w1[j] = load_slice_nt<DT>(wrow[j], (size_t)(two ? s1 : s0)); }
#pragma unroll
      for (int r = 0; r < MR; r++) {
        const f32x4* xp = reinterpret_cast<const f32x4*>(a.A + (size_t)min(r, M - 1) * a.lda);
        f32x4 xa = xp[2 * s0], xb = xp[2 * s0 + 1], ya = xp[2 * (two ? s1 : s0)], yb = xp[2 * (two ? s1 : s0) + 1];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          xa[i] = round_storage_if<DT>(xa[i], a.terms == 1); xb[i] = round_storage_if<DT>(xb[i], a.terms == 1);
          ya[i] = two ? round_storage_if<DT>(ya[i], a.terms == 1) : 0.f; yb[i] = two ? round_storage_if<DT>(yb[i], a.terms == 1) : 0.f;
        }
#pragma unroll
        for (int j = 0; j < NC; j++) { acc[s][j][r] = dot8<DT>(acc[s][j][r], w0[j], xa, xb); acc[s][j][r] = dot8<DT>(acc[s][j][r], w1[j], ya, yb); }
      }
    }
  }
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int j = 0; j < NC; j++)
#pragma unroll
      for (int r = 0; r < MR; r++) {
        const float v = wave_sum(acc[s][j][r]);
        if (lane == 0) s_part[wv][(s * MR + r) * NC + j] = v;
      }
  __syncthreads();
  const int r = threadIdx.x / NC, j = threadIdx.x % NC, n = n0 + j;
  if (r < MR && r < M && n < N) {
    float* cp = g.p[0].C + (size_t)r * g.p[0].ldc + n;
    float v = *cp;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const int at = (s * MR + r) * NC + j;
      v = fmaf(s_part[0][at] + s_part[1][at] + s_part[2][at] + s_part[3][at], g.p[s].scale, v);
    }
    *cp = v;
  }
}

}  // namespace tgx
