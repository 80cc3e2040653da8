// stack_latent.h — a latent attention's values from the records of its divided keys, for steps of few tokens: latent_attn_merge_kernel (stack.h) and the product
// o[t][h] = (lat[t][h] . uv[h]^T) * sigmoid(gate) behind it (stack_gemm.h, SG_GATE) in one launch.
// What bounds it is the launch and two round trips: a workgroup, 32 columns of one head and one token, asks for its weights and, each wave a quarter of the channels, for every record at
// once, merges these into LDS and multiplies.  A head's workgroups merge the same records again: 15 KB each from L2 instead of a launch.  Eight heads of 256 x 128, us: four tokens
// of 15 records 4.5, two of 17 5.1, where merge and product were 4.5 + 4.5 and 4.4 + 4.6; with four tokens a workgroup (60 loads a wave) 8.0.
// Nothing is rounded: the merged rows stay in 32 bits.  Ranks of whole 64s up to LATV_MAX_RANK; a record's row may be longer than the rank that is multiplied (a rotated key part).
#pragma once
#include "stack.h"
#include "stack_gemm.h"

namespace tgx {

constexpr int LATV_MAX_RANK = 512, LATV_COLS = 32;
template <int DT>
__global__ __launch_bounds__(256) void latent_values_kernel(const LatentAttnArgs a, const StackGemmArgs g) {
  constexpr int NS = LATV_MAX_RANK / 64, KC = LATV_MAX_RANK / 256, RECS = 16;      // slices of eight channels a thread multiplies, channels a lane merges, records at once
  __shared__ __attribute__((aligned(16))) float s_lat[LATV_MAX_RANK];
  const int t = blockIdx.z, h = blockIdx.y, n0 = blockIdx.x * LATV_COLS, tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = tid >> 3, part = tid & 7, n = min(n0 + col, g.N - 1), nsl = g.K >> 3, per = g.K >> 2, c0 = wv * per;
  const elem_t<DT>* wr = reinterpret_cast<const elem_t<DT>*>(g.B) + (size_t)h * g.b_zstride + (size_t)n * g.ldb;
  Slice8<DT> w[NS];
#pragma unroll
  for (int i = 0; i < NS; i++) if (8 * i < nsl) w[i] = load_slice_nt<DT>(wr, (size_t)(part + 8 * i));      // (whole 64s: no slice past the end)
  const float gate = g.G[(size_t)t * g.ldg + g.g_col0 + (g.g_per_z ? (size_t)h : (size_t)h * g.c_zoff + n)];
  const size_t rs = (size_t)(a.rank + 2);
  const float* rec = a.part + ((size_t)t * a.heads + h) * a.nsplit * rs;
  const float ms = lane < a.nsplit ? rec[(size_t)lane * rs] : -INFINITY, ls = lane < a.nsplit ? rec[(size_t)lane * rs + 1] : 0.f;      // (at most 64 records)
  float v[KC];
#pragma unroll
  for (int k = 0; k < KC; k++) v[k] = 0.f;
  float f = 0.f, inv = 0.f;
  for (int s0 = 0; s0 < a.nsplit; s0 += RECS) {
    float x[RECS][KC];
#pragma unroll
    for (int s = 0; s < RECS; s++)
#pragma unroll
      for (int k = 0; k < KC; k++) if (64 * k < per) x[s][k] = rec[(size_t)min(s0 + s, a.nsplit - 1) * rs + 2 + c0 + min(64 * k + lane, per - 1)];
    if (s0 == 0) {
      const float M = group_max<64>(ms);
      f = ms == -INFINITY ? 0.f : expf(ms - M);
      const float L = group_sum<64>(ls * f);
      inv = L > 0.f ? 1.0f / L : 0.f;
    }
#pragma unroll
    for (int s = 0; s < RECS; s++) {
      if (s0 + s >= a.nsplit) break;
      const float fs = __uint_as_float((unsigned int)__builtin_amdgcn_readlane((int)__float_as_uint(f), s0 + s));
#pragma unroll
      for (int k = 0; k < KC; k++) if (64 * k < per) v[k] = fmaf(x[s][k], fs, v[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < KC; k++) if (64 * k + lane < per) s_lat[c0 + 64 * k + lane] = v[k] * inv;
  __syncthreads();
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < NS; i++) {
    const int s = part + 8 * i;
    if (8 * i < nsl) acc = dot8<DT>(acc, w[i], *reinterpret_cast<const f32x4*>(&s_lat[8 * s]), *reinterpret_cast<const f32x4*>(&s_lat[8 * s + 4]));
  }
  acc = row_group_sum<8>(acc);
  if (part == 0 && n0 + col < g.N) g.C[(size_t)t * g.ldc + (size_t)h * g.c_zoff + n] = acc / (1.0f + expf(-gate));
}

}  // namespace tgx
