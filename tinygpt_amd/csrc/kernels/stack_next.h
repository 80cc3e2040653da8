// stack_next.h — what stands between two greedy decode steps of a layered model, in one launch behind the logits' argmax partials (slot_logits_kernel): a row's argmax, the token published as
// finalize_row does (gemv.h), and the next step's inputs: its token, position and state buffer, and in designs whose stream begins as the plain embedding row that row.
//
// The launch is latency alone: it replaces one a row for the token, one for the step's tables and one for the embedding, each 2.4 to 4.6 us where an empty launch is 2.4.  A workgroup of sixteen
// waves owns a row.  (It could go through the row's logits itself and save the partials' launch, but one compute unit would read them.  A step of a small model, us, partials' launch and this
// one / this one over the logits: 8192 columns 38.9 / 47.8, 32768 42.2 / 49.8, 65536 46.3 / 54.3.)
#pragma once
#include "gemv.h"
#include "stack_meta.h"

namespace tgx {

struct StackNextArgs {
  FinalizeArgs f;                          // row 0's view; its x is not written
  long long part_stride;
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
  const float* pv = f.part_val + (size_t)r * a.part_stride;
  const int* pi = f.part_idx + (size_t)r * a.part_stride;
  if (tid == 0) s_e = -1;
  __syncthreads();
  for (int i = tid; i < a.S; i += 1024) if (a.ent_row[i] == r) s_e = i;      // (a slot has one entry at most; one outside the step keeps the partials of its last)
  float bv = -INFINITY; int bi = 0x7fffffff;
  auto take = [&](float v, int i) { if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; } };
  for (int i = tid; i < f.n_part; i += 1024) take(pv[i], pi[i]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) { const float v = __shfl_xor(bv, o, 64); const int i = __shfl_xor(bi, o, 64); take(v, i); }
  if ((tid & 63) == 0) { sv[tid >> 6] = bv; si[tid >> 6] = bi; }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 16; w++) take(sv[w], si[w]);                       // (the same in every thread)
  const int e = s_e;
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
