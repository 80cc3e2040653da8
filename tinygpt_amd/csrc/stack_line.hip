// stack_line.hip — launches of the prompt products of layered models (kernels/stack_line.h); a translation unit of its own so that its template instances compile
// beside stack.hip.
#include "stack.h"

#include "prefill_plan.h"
#include "kernels/stack_line.h"

namespace {
template <int DT, int EPI, bool DUAL, bool SHARED>
void launch_line_t(tgx_ctx* c, const tgx::LineArgs& a, dim3 grid, int tile) {
  if (tile == 256) {
    if (stack_allow_lds(c, (const void*)&tgx::stack_line256_kernel<DT, EPI, DUAL, SHARED>, tgx::LINE256_LDS))
      hipLaunchKernelGGL((tgx::stack_line256_kernel<DT, EPI, DUAL, SHARED>), grid, dim3(512), tgx::LINE256_LDS, c->stream, a);
  } else if (tgx::eight_wave_halves(a.g.K >> 6)) {
    if (stack_allow_lds(c, (const void*)&tgx::stack_line128_kernel<DT, EPI, DUAL, SHARED, true>, tgx::LINE128_LDS))
      hipLaunchKernelGGL((tgx::stack_line128_kernel<DT, EPI, DUAL, SHARED, true>), grid, dim3(512), tgx::LINE128_LDS, c->stream, a);
  } else if (stack_allow_lds(c, (const void*)&tgx::stack_line128_kernel<DT, EPI, DUAL, SHARED, false>, tgx::LINE128_LDS))
    hipLaunchKernelGGL((tgx::stack_line128_kernel<DT, EPI, DUAL, SHARED, false>), grid, dim3(512), tgx::LINE128_LDS, c->stream, a);
}
template <int DT, int EPI, bool DUAL>
void launch_line_t(tgx_ctx* c, const tgx::LineArgs& a, dim3 grid, int tile) {
  if constexpr (EPI != tgx::SG_EXPERT_ACT)      // (of experts alone, whose tiles are whole)
    if (a.cus) { launch_line_t<DT, EPI, DUAL, true>(c, a, grid, tile); return; }
  launch_line_t<DT, EPI, DUAL, false>(c, a, grid, tile);
}
// 256-row or 128-row tiles for t256 / t128 of them: a compute unit takes 2.8 times as long for the large one, between what a lone round shows (2048 x 2048 x 2048: 113 us on 64 tiles of
// 256 x 256, 95 with them halved, 48 on 256 of 128 x 128) and what full ones do (K 2048, gate and up of 8192, 2048 rows: 229 us for two rounds, 290 for eight; of 4096 118 and 149).  A last
// round counts whole where it is halved too (line_plan.h): 2048 x 9344 x 2048, 296 tiles with 40 halved 174 us, 1168 small ones 178.  Fewer than 64 small ones leave most of the chip idle either way: the 64-wide tiles
// (0) spread further (130 rows, 1024 x 1024: 18.7 us against 20.4 with the split)
int tile_of(const tgx_ctx* c, long long t256, long long t128) {
  if (t128 < 64) return 0;
  const long long r256 = (t256 + c->num_cus - 1) / c->num_cus, r128 = (t128 + c->num_cus - 1) / c->num_cus;
  return r256 * 28 <= r128 * 10 ? 256 : 128;
}
// whether there is memory for halved tiles (the step asked for it, reserve_share); option stack.ws_max can forbid what is there
bool share_scratch(const tgx_ctx* c, int tile) {
  const StackModel* sm = c->stack;
  const size_t need = tgx::line_share_elems(tile, c->num_cus);
  return need <= sm->share_elems && (sm->ws_max < 0 || need * sizeof(float) <= (size_t)sm->ws_max * 1024);
}
}  // namespace

int stack_line_tile(const tgx_ctx* c, long long M, long long N, bool dual, int nz) {
  const long long n = dual ? 2 * N : N;
  return tile_of(c, (M + 255) / 256 * ((n + 255) / 256) * nz, (M + 127) / 128 * ((n + 127) / 128) * nz);
}
// a grouped product of `pairs` rows over `groups` experts of equal shares (N: columns of both products of a dual one)
int stack_line_tile_grouped(const tgx_ctx* c, long long pairs, int groups, long long N) {
  const long long avg = (pairs + groups - 1) / groups;
  if (avg < 64) return 0;      // tiles of 128 rows would stand more than half empty
  return tile_of(c, groups * ((avg + 255) / 256) * ((N + 255) / 256), groups * ((avg + 127) / 128) * ((N + 127) / 128));
}

void launch_split_terms(tgx_ctx* c, const float* a, long long lda, int rows, int cols, unsigned short* out) {
  TGX_DT16_SWITCH(c->dt, hipLaunchKernelGGL(tgx::split_terms_kernel<DT>, dim3(rows), dim3(256), 0, c->stream, a, lda, cols, c->act16 ? 1 : 0, out))
}

// terms: lines of ldt elements a row (launch_split_terms, or the lines that the product in front wrote); row_tiles: of `tile` rows (an upper bound for grouped products)
void launch_stack_line(tgx_ctx* c, const tgx::StackGemmArgs& g, int epi, int nz, int tile, int row_tiles, const unsigned short* terms, long long ldt) {
  tgx::LineArgs a{};
  a.g = g; a.terms = terms; a.ldt = ldt; a.gm = row_tiles;
  a.gn = tgx::sg_dual(epi) ? (g.N + tile / 2 - 1) / (tile / 2) : (g.N + tile - 1) / tile;
  int wgs = a.gm * a.gn;
  if (nz == 1 && !g.z_off && c->stack->line_share) {      // (experts' rows stand in any order in their tiles: whole ones give a row the same sum wherever it stands)
    const tgx::LineShare sh = tgx::line_share(wgs, tile, g.K >> 6, c->num_cus);
    if (sh.rest && share_scratch(c, tile)) {
      a.cus = c->num_cus; a.met = reinterpret_cast<int*>(c->stack->share); a.sums = c->stack->share + c->num_cus;
      wgs += sh.rest;
    }
  }
  const dim3 grid((unsigned)wgs, g.z_off ? 1 : nz);
  TGX_DT16_SWITCH(c->dt,
    switch (epi) {
      case tgx::SG_STORE: launch_line_t<DT, tgx::SG_STORE, false>(c, a, grid, tile); break;
      case tgx::SG_ADD: launch_line_t<DT, tgx::SG_ADD, false>(c, a, grid, tile); break;
      case tgx::SG_GATE: launch_line_t<DT, tgx::SG_GATE, false>(c, a, grid, tile); break;
      case tgx::SG_ROWSCALE: launch_line_t<DT, tgx::SG_ROWSCALE, false>(c, a, grid, tile); break;
      case tgx::SG_SILU_MUL: launch_line_t<DT, tgx::SG_SILU_MUL, true>(c, a, grid, tile); break;
      default: launch_line_t<DT, tgx::SG_EXPERT_ACT, true>(c, a, grid, tile); break;
    })
}
