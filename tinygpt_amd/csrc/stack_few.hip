// stack_few.hip — launches of the few-row products of layered models (kernels/stack_few.h); a translation unit of its own so that its template instances compile
// beside stack.hip.
#include "stack.h"

#include "kernels/stack_few.h"

namespace {
constexpr size_t LDS_BYTES = 160 * 1024;

template <int DT, int EPI, bool DUAL, int MB>
void launch_few_mb(tgx_ctx* c, const tgx::StackGemmArgs& a, dim3 grid) {
  // Waves and ring depth: some eight waves a compute unit (2048 on the chip) and four a workgroup at least, never more than K has steps; two steps of each in flight, one
  // where the launch has a thousand workgroups that cover for each other.  Measured, us at waves / depth 4/1, 4/2, 8/1, 8/2, 16/1: sixteen rows 1024 x 1024 (64 workgroups):
  // 6.7, 5.9, 5.6, 5.6, 5.5; eight rows 2048 x 8192 (128): 36.6, 22.7, 23.3, 18.5, 18.8; 4096 x 2048 (256): 12.8, 9.3, 9.8, 8.8, 9.3; 8192 x 2048 (512): 15.1, 13.0, 14.0, 15.5,
  // 15.7; sixteen rows 24576 x 1024 (1536): 16.8, 17.7, 18.1, 26.7, 26.8
  const long long wgs = (long long)grid.x * grid.y * grid.z;
  const int steps = (a.K + 63) / 64;
  int nw = 4;
  while (nw < tgx::few_max_waves(MB) && wgs * nw < 8LL * c->num_cus) nw *= 2;
  while (nw > 1 && nw > steps) nw /= 2;
  int depth = wgs >= 4LL * c->num_cus || nw >= steps ? 1 : 2;
  while (tgx::few_lds_bytes<DT, DUAL, MB>(nw, depth) > LDS_BYTES) { if (depth > 1) depth--; else nw /= 2; }
  const size_t lds = tgx::few_lds_bytes<DT, DUAL, MB>(nw, depth);
  if (!stack_allow_lds(c, (const void*)&tgx::stack_few_kernel<DT, EPI, DUAL, MB>, lds)) return;
  hipLaunchKernelGGL((tgx::stack_few_kernel<DT, EPI, DUAL, MB>), grid, dim3(64 * nw), lds, c->stream, a, depth);
}
template <int DT, int EPI, bool DUAL>
void launch_few_t(tgx_ctx* c, const tgx::StackGemmArgs& a, dim3 grid, int mb) {
  switch (mb) {
    case 1: launch_few_mb<DT, EPI, DUAL, 1>(c, a, grid); break;
    case 2: launch_few_mb<DT, EPI, DUAL, 2>(c, a, grid); break;
    default: launch_few_mb<DT, EPI, DUAL, 4>(c, a, grid); break;
  }
}
}  // namespace

void launch_stack_few(tgx_ctx* c, const tgx::StackGemmArgs& a, int epi, int nz, int dt) {
  // sixteen-row operands: all rows of a step in one workgroup up to 64 (the weights cross once); many rows of a narrow matrix (a router's) in sixteens, which spreads
  // them over the chip
  const int mb = a.M <= 16 || a.M > 64 ? 1 : a.M <= 32 ? 2 : 4;
  const dim3 grid((a.N + 15) / 16, (a.M + 16 * mb - 1) / (16 * mb), nz);
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
