// prefill_plan.h — how a prompt's products are cut, as plain arithmetic on their sizes (no HIP: tests/test_prefill_plan.py goes through it on the CPU).
#pragma once

namespace tgx {

// K (a multiple of 64) in z slabs: steps of 64 in each but the last, and whether the last one has any.  (Rounding up can leave none for it: 25 steps in six slabs are five of five.)
inline int slab_steps(int K, int z) { return (K / 64 + z - 1) / z; }
inline bool slabs_hold_k(int K, int z) { return (z - 1) * slab_steps(K, z) < K / 64; }

// Slabs of an N = hidden product on the eight-wave 128 x 128 kernel (1: whole).  Slabs z = 2..8 that shorten the critical path: rounds of workgroups x 1 / z of the K loop against one
// round of whole tiles (160 tiles on 256 CUs: z = 3 -> 2 rounds of a third = 0.67; 128 tiles: z = 2 -> 0.5); taken from 0.8 down (the slabs cost a pass over z x M x N floats).  More
// than four where all of them run at once and the steps of K that they save (0.6 us each) outweigh their floats (written and read at 5 TB/s): eight / four, ms per prompt,
// Llama-3.2-1B 133 tokens 2.14 / 2.25, 256 2.28 / 2.39, Qwen2.5-0.5B 256 2.51 / 2.67; with eight in two rounds or for K 2048 at 509 rows and N 1024 it is slower
// (Qwen3-0.6B 3.53 / 3.45).  From 385 rows on the sixth to eighth slab costs its reader more (Qwen3-0.6B, K 3072, eight / as few as that takes: 400 tokens 3.03 / 2.97, 450 3.13 / 2.95,
// 509 3.22 / 3.08, 600 3.58 / 3.53; 330 2.84 / 2.87).  Every slab has four steps on average and one at least.
inline int eight_wave_slabs(int M, int N, int K, int num_cus) {
  const int tiles = ((N + 127) / 128) * ((M + 127) / 128);
  int z = 1;
  double best = 0.8001;
  for (int zz = 2; zz <= 8 && tiles < num_cus; zz++) {
    if (zz > 4 && (zz * tiles > num_cus || K < (zz > 5 && M > 384 ? 1e-3 : 6.8e-4) * zz * M * N)) break;
    const double cost = (double)((zz * tiles + num_cus - 1) / num_cus) / zz;
    if (cost < best - 1e-9 && K / 64 >= 4 * zz && slabs_hold_k(K, zz)) { best = cost; z = zz; }
  }
  return z;
}

// Whether the gate_up product (N columns, below a chip of 128 x 128 tiles) of a prompt stays whole on the eight-wave kernel instead of K slabs with a launch that sums them.  most: the
// half-chips of tiles up to which that kernel is taken (option prefill.wide_8k_max).  A whole product is a chain of K / 64 steps of 0.6 us, so a short K keeps it from a quarter of a
// chip of tiles on, a longer one from half a chip on, where slabs would go into another round.  Whole / split, ms per prompt: Qwen3-0.6B (K 1024) 133 tokens (96 tiles) 2.68 / 2.78, 256
// 2.98 / 3.21, 509 (192) 3.45 / 3.92; Qwen2.5-0.5B 133 (152) 2.07 / 2.27, 384 (228) 2.49 / 2.99.  Whole less split, us a layer: K 512 and 1024, 129 to 512 rows, 64 to 240 tiles -0.7 to
// -21; K 2048, 129 to 512 rows, 64 tiles +5 to +7, 96 -4 to +2, 128 -3 to 0, 144 to 240 -14 to -28; K 2560, 3072 and 4096, 65 to 200 rows, 64 tiles +14 to +21, 96 -2 to +2, 128 +1 to
// +7, 152 -8 to -18, 192 -17 to -33, 224 -20 to -37 (profiles/prompt_gate_up_whole.txt).  Up to 64 rows the slabs have tiles of 64 rows and nothing of it is padding.
inline bool gate_up_whole(int M, int N, int K, int num_cus, int most) {
  const long long tiles = (long long)((N + 127) / 128) * ((M + 127) / 128);
  if (M <= 64 || tiles >= num_cus || 2 * tiles > (long long)most * num_cus) return false;
  return K <= 1024 && M > 128 ? 4 * tiles >= num_cus : 2 * tiles > num_cus;
}

// Whether the eight waves of a 128 x 128 tile divide a stage of K into halves (gemm_dma8h_kernel, both sides' times there) and not into quarters: chains of few stages, which are mostly
// what stands in front of and behind them.
inline bool eight_wave_halves(int stages) { return stages <= 32; }

}  // namespace tgx
