// stack_rec_args.h — what a recurrence over a portion's tokens takes, whichever form runs it (stack_rec.h: token by token; stack_rec_block.h: in blocks).
#pragma once

namespace tgx {

enum { REC_WKV = 0, REC_DELTA = 1, REC_SSD = 2, REC_CDELTA = 3 };
struct RecScanArgs {
  const float* a; long long lda;     // per token and key head [dim]: the read vector (wkv: r, delta: q, ssd: C)
  const float* k; long long ldk;     //                               k (ssd: B)
  const float* w; long long ldw;     //                               wkv: the decay per channel; cdelta: per (query) head and channel
  const float* v; long long ldv;     // per token and head [vdim]
  const float* beta; const float* g; long long ldg;      // delta, ssd: per token and head (cdelta: beta alone)
  const float* fixed; float beta0;   // ssd: [heads] decays that hold for every token, with beta0 as every token's beta (nullptr: beta and g)
  const float* u;                    // wkv: [heads][dim] bonus
  const float* skip;                 // ssd: [heads] (nullptr: none)
  float* S;                          // [slots][heads][dim][vdim]
  float* out; long long ldo;         // [T][heads * vdim]
  int heads, kv_heads, dim, vdim;
};
constexpr int REC_BLOCK = 32, REC_BLOCK_MAX_DIM = 128, REC_BLOCK_MAX_VDIM = 256;      // tokens of a block; the largest head that blocks take

}  // namespace tgx
