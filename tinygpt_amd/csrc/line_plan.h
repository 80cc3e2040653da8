// line_plan.h — how the last tiles of a prompt's product (kernels/stack_line.h) are divided between the compute units, as plain arithmetic on their number (no HIP call: tests go
// through it on the CPU, the kernels through the same function).
#pragma once
#include <cstddef>

#if defined(__HIPCC__)
#define TGX_HD __host__ __device__ inline
#else
#define TGX_HD inline
#endif

namespace tgx {

// Whole tiles in rounds of one workgroup a compute unit, then `rest`, at most half a round, each as two halves of its steps of K (64 each); rest 0: every tile is whole.
struct LineShare { int whole, rest; };

// Halving takes half of a tile's steps off the last round and costs a pass of the first half's sums through memory (256 KB a tile of 256 x 256) and a ring filled anew.  From these steps
// on it was faster, us halved / whole: 256 x 256, 10917 x 2048 (88 tiles of 344 halved) K 1024 104 / 108, 2048 170 / 189, 4096 315 / 357, 8192 589 / 685; 10917 x 8192 (96 of 1376)
// K 2048 587 / 602; 2048 x 10240 (64 of 320) 169 / 189.  128 x 128, 1999 x 1024 (128 of 128) K 1024 25.0 / 22.4, 1536 28.1 / 28.6, 2048 31.8 / 34.0, 3072 40.0 / 47.5, 4096 46.2 / 59.1;
// 1999 rows, gate and up of 1536 (128 of 384) K 1024 43.2 / 41.2, 1536 55.2 / 56.2, 2048 66.0 / 70.3, 3072 91.4 / 97.6: at 24 steps the two are within two runs of one.  Beyond half a round two halves are two rounds, and thirds to sevenths lose to the sums' way through memory what
// they save (344 tiles, K 8192: thirds 663, fifths 626; 200 tiles, K 2048: 98 whole, 149 and 174).  The card's power sets the rate of full rounds, so that a half-empty one is not
// half lost.
constexpr int LINE_SHARE_STEPS256 = 16, LINE_SHARE_STEPS128 = 32;
TGX_HD LineShare line_share(int tiles, int tile, int nk, int cus) {
  const int rest = cus > 0 ? tiles % cus : 0;
  return rest && 2 * rest <= cus && nk >= (tile == 256 ? LINE_SHARE_STEPS256 : LINE_SHARE_STEPS128) ? LineShare{tiles - rest, rest} : LineShare{tiles, 0};
}
// floats of a launch's halved tiles: who has come and whose sums lie ready, two numbers for each of half a round at most, then the sums (256 x 256: 128 KB a compute unit)
TGX_HD size_t line_share_elems(int tile, int cus) { return (size_t)cus + (size_t)(cus / 2) * tile * tile; }
// the larger tile of which products of up to `rows` rows, `cols` columns (of both matrices of a dual one) and nk steps can come to halve a round; 0: none.  256 x 256 tiles are taken only
// where those of 128 x 128 are more than two rounds (tile_of, stack_line.hip)
TGX_HD int line_share_tile(long long rows, long long cols, int nk, int cus) {
  if (nk >= LINE_SHARE_STEPS256 && ((rows + 127) / 128) * ((cols + 127) / 128) > 2LL * cus) return 256;
  return nk >= LINE_SHARE_STEPS128 ? 128 : 0;
}

}  // namespace tgx
