// stack_next.h — what stands between two greedy decode steps of a layered model, in one launch: a row's argmax, the token published as finalize_row does (gemv.h), and the next step's
// inputs: its token, position and state buffer, and in designs whose stream begins as the plain embedding row that row.
//
// The launch is latency alone: it replaces one of the argmax partials, one a row for the token, one for the step's tables and one for the embedding, each 2.2 to 4.6 us of which 2.2 is an
// empty launch.  A workgroup of sixteen waves owns a row.  With `scan` it goes through the row's logits itself (NEXT_SCAN), all loads of a lane on their way at once, and leaves the
// partials as slot_logits_kernel would, the row's best in the first of them; otherwise it starts from the partials that are there.
#pragma once
#include "gemv.h"
#include "stack_meta.h"

namespace tgx {

struct StackNextArgs {
  FinalizeArgs f;                          // row 0's view; its x is not written
  long long part_stride;
  float* part_val; int* part_idx;          // all rows' partials
  const float* logits; int scan;           // [rows][V]
  int *tok_id, *tok_pos, *tok_par, *ent_par; const int* ent_row; int S;      // of the step's entries, one token each
  float* x; int W;                         // the next step's stream [S][W]; nullptr: the design's own launch begins it
};
template <int DT>
__global__ __launch_bounds__(1024) void stack_next_kernel(const StackNextArgs a) {
  __shared__ float sv[16];
  __shared__ int si[16], s_e;
  const int r = blockIdx.x, tid = threadIdx.x;
  FinalizeArgs f = a.f;
  f.tok += r; f.pos += r; f.row = a.f.row + r;
  float* pv = a.part_val + (size_t)r * a.part_stride;
  int* pi = a.part_idx + (size_t)r * a.part_stride;
  if (tid == 0) s_e = -1;
  __syncthreads();
  for (int i = tid; i < a.S; i += 1024) if (a.ent_row[i] == r) s_e = i;      // (a slot has one entry at most)
  float bv; int bi;
  auto take = [&](float v, int i) { if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; } };
  auto best = [&](auto each) {      // over the workgroup, the same in every thread
    bv = -INFINITY; bi = 0x7fffffff;
    each();
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { const float v = __shfl_xor(bv, o, 64); const int i = __shfl_xor(bi, o, 64); take(v, i); }
    if ((tid & 63) == 0) { sv[tid >> 6] = bv; si[tid >> 6] = bi; }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 16; w++) take(sv[w], si[w]);
  };
  const float* lg = a.logits + (size_t)r * f.V;
  if (a.scan) best([&] {            // (asked for before it is known whether the slot takes part)
    if ((f.V & 3) == 0) {
      const int n4 = f.V >> 2;
      for (int i0 = tid; i0 < n4; i0 += 8 * 1024) {
        f32x4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = reinterpret_cast<const f32x4*>(lg)[min(i0 + 1024 * u, n4 - 1)];      // (past the end: the last again, which changes no maximum)
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
          for (int j = 0; j < 4; j++) take(v[u][j], 4 * min(i0 + 1024 * u, n4 - 1) + j);
      }
    } else
      for (int i = tid; i < f.V; i += 1024) take(lg[i], i);
  });
  else __syncthreads();
  const int e = s_e;
  const bool scan = a.scan && e >= 0;      // a slot outside the step keeps the partials of its last one
  if (!scan) {
    __syncthreads();                       // (sv and si are read)
    best([&] { for (int i = tid; i < f.n_part; i += 1024) take(pv[i], pi[i]); });
  } else
    for (int p = tid; p < f.n_part; p += 1024) { pv[p] = p == 0 ? bv : -INFINITY; pi[p] = p == 0 ? bi : 0x7fffffff; }
  if (e >= 0 && a.x) {
    const int t = (unsigned)bi < (unsigned)f.V ? bi : 0;
    const elem_t<DT>* row = static_cast<const elem_t<DT>*>(f.embed) + (size_t)t * a.W;
    for (int c = tid; c < a.W; c += 1024) a.x[(size_t)e * a.W + c] = elem_to_f32<DT>(row[c]);
  }
  if (tid == 1023) {                       // (the last wave: the row's load of a narrow stream is not behind this)
    int t, pos;
    publish_token(f, bi, t, pos);
    if (e >= 0) { a.tok_id[e] = t; a.tok_pos[e] += 1; a.ent_par[e] ^= 1; a.tok_par[e] ^= 1; }
  }
}

}  // namespace tgx
