// stack_few.hip — launches of the few-row products of layered models (kernels/stack_few.h); a translation unit of its own so that its template instances compile
// beside stack.hip.
#include "stack.h"

#include "kernels/stack_few.h"

namespace {
template <int DT, int EPI, bool DUAL, int MB, int XP>
void launch_few_mb(tgx_ctx* c, const tgx::StackGemmArgs& a, dim3 grid) {
  const tgx::FewPlan p = tgx::few_plan<DT, DUAL, MB, XP>(c->num_cus, (long long)grid.x * grid.y * grid.z, a.K);
  if (!stack_allow_lds(c, (const void*)&tgx::stack_few_kernel<DT, EPI, DUAL, MB, XP>, p.lds)) return;
  hipLaunchKernelGGL((tgx::stack_few_kernel<DT, EPI, DUAL, MB, XP>), grid, dim3(64 * p.nw), p.lds, c->stream, a, p.depth);
}
template <int DT, int MB, int XP>
void launch_few_pair_mb(tgx_ctx* c, const tgx::StackGemmArgs& a, const tgx::StackGemmArgs& b, dim3 grid) {
  const tgx::FewPlan p = tgx::few_plan<DT, false, MB, XP>(c->num_cus, (long long)grid.x * grid.y * grid.z, a.K);
  if (!stack_allow_lds(c, (const void*)&tgx::stack_few_pair_kernel<DT, MB, XP>, p.lds)) return;
  hipLaunchKernelGGL((tgx::stack_few_pair_kernel<DT, MB, XP>), grid, dim3(64 * p.nw), p.lds, c->stream, a, b, p.depth);
}
template <int DT, int EPI, bool DUAL>
void launch_few_t(tgx_ctx* c, const tgx::StackGemmArgs& a, dim3 grid, int mb) {
  switch (mb) {
    case 1: {
      const int xp = tgx::few_pieces(a);
      if (xp == 1) launch_few_mb<DT, EPI, DUAL, 1, 1>(c, a, grid);
      else if (xp == 2) launch_few_mb<DT, EPI, DUAL, 1, 2>(c, a, grid);
      else launch_few_mb<DT, EPI, DUAL, 1, 4>(c, a, grid);
      break;
    }
    case 2: launch_few_mb<DT, EPI, DUAL, 2, 4>(c, a, grid); break;
    default: launch_few_mb<DT, EPI, DUAL, 4, 4>(c, a, grid); break;
  }
}
}  // namespace

// two stored products of up to 64 rows, the same for both, and of one contraction length
void launch_stack_few_pair(tgx_ctx* c, const tgx::StackGemmArgs& a, const tgx::StackGemmArgs& b, int dt) {
  const int mb = a.M <= 16 ? 1 : a.M <= 32 ? 2 : 4;
  const dim3 grid((std::max(a.N, b.N) + 15) / 16, 1, 2);
  TGX_DT_SWITCH(dt,
    if (mb == 1 && tgx::few_pieces(a) == 1) launch_few_pair_mb<DT, 1, 1>(c, a, b, grid);
    else if (mb == 1 && tgx::few_pieces(a) == 2) launch_few_pair_mb<DT, 1, 2>(c, a, b, grid);
    else if (mb == 1) launch_few_pair_mb<DT, 1, 4>(c, a, b, grid);
    else if (mb == 2) launch_few_pair_mb<DT, 2, 4>(c, a, b, grid);
    else launch_few_pair_mb<DT, 4, 4>(c, a, b, grid);)
}

// grouped_tiles: upper bound of the tile list of a grouped product (a.z_off), 0 for plain and batched ones
void launch_stack_few(tgx_ctx* c, const tgx::StackGemmArgs& a, int epi, int nz, int grouped_tiles, int dt) {
  // sixteen-row operands: all rows of a step in one workgroup up to 64 (the weights cross once); many rows of a narrow matrix (a router's) in sixteens, which spreads
  // them over the chip
  const int mb = a.z_off || a.M <= 16 || a.M > 64 ? 1 : a.M <= 32 ? 2 : 4;
  const dim3 grid((a.N + 15) / 16, a.z_off ? grouped_tiles : (a.M + 16 * mb - 1) / (16 * mb), a.z_off ? 1 : nz);
  TGX_DT_SWITCH(dt,
    switch (epi) {
      case tgx::SG_STORE: launch_few_t<DT, tgx::SG_STORE, false>(c, a, grid, mb); break;
      case tgx::SG_ADD: launch_few_t<DT, tgx::SG_ADD, false>(c, a, grid, mb); break;
      case tgx::SG_GATE: launch_few_t<DT, tgx::SG_GATE, false>(c, a, grid, mb); break;
      case tgx::SG_ROWSCALE: launch_few_t<DT, tgx::SG_ROWSCALE, false>(c, a, grid, mb); break;
      case tgx::SG_SILU_MUL: launch_few_t<DT, tgx::SG_SILU_MUL, true>(c, a, grid, mb); break;
      default: launch_few_t<DT, tgx::SG_EXPERT_ACT, true>(c, a, grid, mb); break;
    })
}
