// stack_ssd.hip — launches of the blocked scalar-decay state-space recurrence on the matrix cores (kernels/stack_ssd_mfma.h); a translation unit of its own so that its
// template instances compile beside stack.hip.
#include "stack.h"

#include "kernels/stack_ssd_mfma.h"

bool ssd_mfma_shapes_ok(int heads, int groups, int N, int E, long long ld) { return N % 4 == 0 && N <= 256 && (heads * E) % 4 == 0 && ld % 4 == 0 && ld < (1 << 21) && groups > 0; }
size_t ssd_gram_elems(int T, int S, int groups) { return ((size_t)T / tgx::SSD_BLOCK + (size_t)S + 1) * groups * tgx::SSD_BLOCK * tgx::SSD_BLOCK; }

namespace {
int ssd_tiles(int E, bool norm) { return (E + 31) / 32 + (norm ? 1 : 0); }
int ssd_state_tiles(int N) { return N <= 128 ? 1 : 2; }
int ssd_room(const tgx_ctx* c, int N) { return (ssd_state_tiles(N) == 1 ? 2 : 1) * c->num_cus; }      // workgroups that run at once: two a compute unit, one above 128 channels
}  // namespace
// Blocks of a portion (0: entries whole).  As many portions as the chip has room for beside the entries' heads, of two blocks at least, from six blocks on.
// A prompt of 8 heads of 128 x 256, whole and in two launches: four blocks 29.6 us and 29.4 with a launch more, eight 54 and 37, sixteen 105 and 54, 32 212 and 80.
// Two workgroups on a compute unit take half as long again a block as one, and the states' launch is half of the portions', so with room for two portions only nothing is won where that is two
// a compute unit (4 heads of 128 x 256, eight entries of seven blocks 49 and 62; 16 heads, two of sixteen 101 and 108; 32 heads, one of 32 197 and 192), and three need eight blocks
// (16 heads of 128 x 256 with a second state: one entry of seven 48 and 49, of eight 55 and 49).  Above 128 channels two are enough (16 heads of 256 x 256, one entry: seven blocks 69 and 64, 32 289 and 208).
int ssd_portion(const tgx_ctx* c, int S, int heads, int N, int E, bool norm, int max_count) {
  const long long whole = (long long)S * heads * ssd_tiles(E, norm), most = ssd_room(c, N) / whole;
  const int blocks = (max_count + tgx::SSD_BLOCK - 1) / tgx::SSD_BLOCK, least = ssd_state_tiles(N) > 1 ? 2 : blocks < 8 ? 4 : 3;
  if (blocks < 6 || most < least) return 0;
  const int P = (int)std::min<long long>(most, blocks / 2);
  return (blocks + P - 1) / P;
}
size_t ssd_portion_elems(int S, int heads, int N, int E, bool norm, int max_count, int portion) {
  const int blocks = (max_count + tgx::SSD_BLOCK - 1) / tgx::SSD_BLOCK;
  return portion ? (size_t)S * ((blocks + portion - 1) / portion) * heads * ssd_tiles(E, norm) * tgx::ssd_state_elems(ssd_state_tiles(N)) : 0;
}
// the most that is: room for so many workgroups
size_t ssd_portion_most(const tgx_ctx* c) { return 2 * (size_t)c->num_cus * tgx::ssd_state_elems(1); }

void launch_ssd_mfma(tgx_ctx* c, const tgx::StepMeta& m, tgx::SsdArgs a, int S, int max_count) {
  if (!ssd_mfma_shapes_ok(a.heads, a.groups, a.N, a.E, a.ld) || a.b0 % 4 || a.c0 % 4) { c->launch_fault = "blocked state-space recurrence: sizes it does not take"; return; }
  const int blocks = (max_count + tgx::SSD_BLOCK - 1) / tgx::SSD_BLOCK;
  hipLaunchKernelGGL(tgx::ssd_gram_kernel<>, dim3(blocks, a.groups, S), dim3(256), 0, c->stream, m, a);
  a.portions = a.portion ? (blocks + a.portion - 1) / a.portion : 1;
  const dim3 grid(a.heads, ssd_tiles(a.E, a.norm_S), S * a.portions);
  a.ranked = (long long)grid.x * grid.y * S > ssd_room(c, a.N);
  auto go = [&](auto NW, auto NORM, auto MODE) { hipLaunchKernelGGL((tgx::ssd_block_kernel<decltype(NW)::value, decltype(NORM)::value, decltype(MODE)::value>), grid, dim3(256), 0, c->stream, m, a); };
  auto mode = [&](auto NW, auto NORM) {
    if (!a.portion) { go(NW, NORM, std::integral_constant<int, tgx::SSD_WHOLE>{}); return; }
    go(NW, NORM, std::integral_constant<int, tgx::SSD_STATES>{});
    go(NW, NORM, std::integral_constant<int, tgx::SSD_PORTIONS>{});
  };
  auto norm = [&](auto NW) { if (a.norm_S) mode(NW, std::true_type{}); else mode(NW, std::false_type{}); };
  if (ssd_state_tiles(a.N) == 1) norm(std::integral_constant<int, 1>{}); else norm(std::integral_constant<int, 2>{});
}

void launch_gate_scan(tgx_ctx* c, const tgx::StepMeta& m, const tgx::GateScanArgs& a, int S) { hipLaunchKernelGGL(tgx::gate_scan_kernel<>, dim3(S, a.heads), dim3(256), 0, c->stream, m, a); }
