// stack_rows.hip — launches of the products over a step's (token, expert) pairs (kernels/stack_rows.h).
#include <type_traits>

#include "stack.h"

#include "kernels/stack_rows.h"

namespace {
template <int DT, int EPI, bool DUAL>
void launch_rows_t(tgx_ctx* c, const tgx::StackGemmArgs& a, dim3 grid) {
  // two waves a workgroup, four while the chip has room for them (eight waves a compute unit).  us at two / four waves: 1152 workgroups of eight chunks of K 12.1 / 13.9, 1536 of
  // eight (two matrices) 10.8 / 13.0, 576 of twelve 11.5 / 11.8, 512 of twelve 7.8 / 7.4, 512 of sixteen 10.2 / 10.1
  const int nw = (long long)grid.x * grid.y * tgx::ROWS_MAX_WAVES <= 8LL * c->num_cus ? tgx::ROWS_MAX_WAVES : 2;
  hipLaunchKernelGGL((tgx::stack_rows_kernel<DT, EPI, DUAL>), grid, dim3(64 * nw), tgx::rows_lds(nw), c->stream, a);
}
}  // namespace

void launch_stack_rows(tgx_ctx* c, const tgx::StackGemmArgs& a, int epi, int dt) {
  const int cols = tgx::rows_cols(tgx::sg_dual(epi));
  const dim3 grid((a.N + cols - 1) / cols, std::min(a.n_pairs, a.experts), (a.tokens + tgx::ROWS_TILE - 1) / tgx::ROWS_TILE);
  TGX_DT_SWITCH(dt,
    switch (epi) {
      case tgx::SG_STORE: launch_rows_t<DT, tgx::SG_STORE, false>(c, a, grid); break;
      case tgx::SG_ROWSCALE: launch_rows_t<DT, tgx::SG_ROWSCALE, false>(c, a, grid); break;
      case tgx::SG_SILU_MUL: launch_rows_t<DT, tgx::SG_SILU_MUL, true>(c, a, grid); break;
      case tgx::SG_EXPERT_ACT: launch_rows_t<DT, tgx::SG_EXPERT_ACT, true>(c, a, grid); break;
      default: c->launch_fault = "grouped product: an epilogue that no expert layer has"; break;
    })
}
