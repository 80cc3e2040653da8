// stack_recblk.hip — launches of the recurrences in blocks of 32 tokens (kernels/stack_rec_block.h).
#include <type_traits>

#include "stack.h"

#include "kernels/stack_rec_block.h"

size_t rec_block_elems(size_t blocks, int heads, int dim, int vdim, bool solve) { return blocks * (size_t)heads * tgx::RecBlockLayout(dim, vdim, solve).stride; }

void launch_rec_blocks(tgx_ctx* c, const tgx::StepMeta& m, const tgx::RecScanArgs& a, int kind, int S, int max_count, float* scratch) {
  const int nblk = (max_count + tgx::REC_BLOCK - 1) / tgx::REC_BLOCK;
  auto go = [&](auto K, auto D) {
    constexpr int KIND = decltype(K)::value, NT = decltype(D)::value;
    hipLaunchKernelGGL((tgx::rec_block_prep_kernel<KIND, 64 * NT>), dim3(nblk, a.heads, S), dim3(256), 0, c->stream, m, a, scratch);
    const dim3 grid(S, a.heads, (a.vdim + 15) / 16);
    hipLaunchKernelGGL((tgx::rec_block_kernel<KIND, NT>), grid, dim3(256), 0, c->stream, m, a, scratch);
  };
  auto dims = [&](auto K) { if (a.dim <= 64) go(K, std::integral_constant<int, 1>{}); else go(K, std::integral_constant<int, 2>{}); };
  if (kind == tgx::REC_WKV) dims(std::integral_constant<int, tgx::REC_WKV>{});
  else if (kind == tgx::REC_CDELTA) dims(std::integral_constant<int, tgx::REC_CDELTA>{});
  else dims(std::integral_constant<int, tgx::REC_DELTA>{});
}
