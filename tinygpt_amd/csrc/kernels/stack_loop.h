// stack_loop.h — row-wise kernels of the layered designs with layer norms (weight and bias) before and after every sublayer, a looped span of layers and
// un-normalised sigmoid attention whose weights are mixed across heads (Zaluvik).  Same conventions as stack.h / stack_seq.h: a step's T tokens are the
// concatenated entries of a ragged batch (StepMeta), all arithmetic here is fp32, every reduction has a fixed order.
//   embed_scale_rows_kernel    x[t] = embed[id] * scale, and a second copy for the loop's re-injection
//   copy_rows_kernel           rows of one width between buffers of different strides
//   layer_norm_rows_kernel     (row - mean) / sqrt(var + eps) * w + b
//   affine_seam_kernel         x += mult * LN_b(sublayer output) and the next sublayer's LN_a input, the experts' combine folded in
//   sigmoid_mix_attn_kernel    a token against the window of its keys in the pool: sigmoid(score + bias) per head, weights mixed across heads, value sums
//   sigmoid_mix_merge_kernel   adds up the partial sums of a window divided between workgroups, applies the output gate
//   (kernels/stack_mix_mfma.h holds the same attention for portions of prompts on the matrix cores)
#pragma once
#include "stack_seq.h"

namespace tgx {

template <int DT>
__global__ __launch_bounds__(256) void embed_scale_rows_kernel(StepMeta m, const elem_t<DT>* embed, float scale, float* x, float* x0, long long ldx0, int W) {
  const int t = blockIdx.x;
  const size_t id = (size_t)m.tok_id[t];
  for (int c = threadIdx.x; c < W; c += 256) {
    const float v = elem_to_f32<DT>(embed[id * W + c]) * scale;
    x[(size_t)t * W + c] = v;
    if (x0) x0[(size_t)t * ldx0 + c] = v;
  }
}

__global__ __launch_bounds__(256) void copy_rows_kernel(const float* src, long long lds, float* dst, long long ldd, int W) {
  const size_t t = blockIdx.x;
  for (int c = threadIdx.x; c < W; c += 256) dst[t * ldd + c] = src[t * lds + c];
}

// mean and 1 / sqrt(variance + eps) of one row, the variance as the mean of the squared deviations (second pass over the row)
__device__ __forceinline__ void row_moments_256(const float* r, int W, float eps, float* s4, float& mean, float& rstd) {
  float s = 0.f;
  for (int c = threadIdx.x; c < W; c += 256) s += r[c];
  mean = block_sum_256(s, s4) / (float)W;
  float q = 0.f;
  for (int c = threadIdx.x; c < W; c += 256) { const float d = r[c] - mean; q = fmaf(d, d, q); }
  rstd = 1.0f / sqrtf(block_sum_256(q, s4) / (float)W + eps);
}

// out[i] = LN(x[rows ? rows[i] : i]) * w + b
__global__ __launch_bounds__(256) void layer_norm_rows_kernel(const float* x, const int* rows, const float* w, const float* b, float* out, int W, float eps) {
  __shared__ float s4[4];
  const float* xr = x + (size_t)(rows ? rows[blockIdx.x] : blockIdx.x) * W;
  float mean, rstd;
  row_moments_256(xr, W, eps, s4, mean, rstd);
  for (int c = threadIdx.x; c < W; c += 256) out[(size_t)blockIdx.x * W + c] = fmaf((xr[c] - mean) * rstd, w[c], b[c]);
}

// ---- the seam between two sublayers of a layer-norm design.  y_t = the sublayer's output for token t: one row, or the sum over the token's `top` expert
// rows (router weights already applied) plus the shared expert's row.  x_t <- x_t + mult * (LN(y_t) * w_post + b_post);  out_t = LN(x_t) * w_next + b_next
// (the next sublayer's input; skipped without w_next: the stream is changed before the next norm, or the model ends).  One workgroup per token.
struct AffineSeamArgs {
  float* x;                  // [T][W]
  const float* y;            // [T * top][W]
  int top;
  const float* ysh;          // [T][W] (nullptr: no shared expert)
  float* ytmp;               // [T][W] scratch
  const float *w_post, *b_post;
  float mult;
  const float *w_next, *b_next;
  float* out;                // [T][W]
  int W; float eps;
};
// Up to a width of 4096 a token's row stays in registers and every load of the seam is on its way before the first of its four sums.  NR vectors a thread, and not
// more than the width needs: a prompt wants the waves (1024 channels, the median launch of two decoded rows 6.5 -> 3.7 us, a
// prompt of 2000 21 -> 13, and 34 with all four vectors' registers held).
template <bool V4, int NR>
__device__ __forceinline__ void affine_seam_row(const AffineSeamArgs& a, size_t t, float (*s4)[4]) {
  float* xt = a.x + t * a.W;
  f32x4 v[NR], xv[NR], wp[NR], bp[NR], wn[NR], bn[NR];
  auto each = [&](auto f) {
#pragma unroll
    for (int k = 0; k < NR; k++)
#pragma unroll
      for (int u = 0; u < 4; u++) if (row_channel<V4>(k, u) < a.W) f(k, u);
  };
#pragma unroll
  for (int k = 0; k < NR; k++) v[k] = row_load<V4>(a.y + t * a.top * a.W, k, a.W);
#pragma unroll
  for (int k = 0; k < NR; k++) { xv[k] = row_load<V4>(xt, k, a.W); wp[k] = row_load<V4>(a.w_post, k, a.W); bp[k] = row_load<V4>(a.b_post, k, a.W); }
  auto add = [&](const float* r) {
#pragma unroll
    for (int k = 0; k < NR; k++) { const f32x4 z = row_load<V4>(r, k, a.W); for (int u = 0; u < 4; u++) v[k][u] += z[u]; }
  };
#pragma unroll 4
  for (int j = 1; j < a.top; j++) add(a.y + (t * a.top + j) * a.W);
  if (a.ysh) add(a.ysh + t * a.W);
  if (a.w_next)
#pragma unroll
    for (int k = 0; k < NR; k++) { wn[k] = row_load<V4>(a.w_next, k, a.W); bn[k] = row_load<V4>(a.b_next, k, a.W); }
  float s = 0.f, q = 0.f;
  each([&](int k, int u) { s += v[k][u]; });
  float mean = block_sum_once(s, s4[0]) / (float)a.W;
  each([&](int k, int u) { const float d = v[k][u] - mean; q = fmaf(d, d, q); });
  float rstd = 1.0f / sqrtf(block_sum_once(q, s4[1]) / (float)a.W + a.eps);
  s = 0.f; q = 0.f;
  each([&](int k, int u) { v[k][u] = fmaf(a.mult, fmaf((v[k][u] - mean) * rstd, wp[k][u], bp[k][u]), xv[k][u]); s += v[k][u]; });
#pragma unroll
  for (int k = 0; k < NR; k++) row_store<V4>(xt, k, a.W, v[k]);
  if (!a.w_next) return;
  mean = block_sum_once(s, s4[2]) / (float)a.W;
  each([&](int k, int u) { const float d = v[k][u] - mean; q = fmaf(d, d, q); });
  rstd = 1.0f / sqrtf(block_sum_once(q, s4[3]) / (float)a.W + a.eps);
#pragma unroll
  for (int k = 0; k < NR; k++) {
    f32x4 o;
#pragma unroll
    for (int u = 0; u < 4; u++) o[u] = fmaf((v[k][u] - mean) * rstd, wn[k][u], bn[k][u]);
    row_store<V4>(a.out + t * a.W, k, a.W, o);
  }
}
template <int NR>
__device__ __forceinline__ void affine_seam_body(AffineSeamArgs a) {
  __shared__ float s44[4][4];
  const size_t t = blockIdx.x;
  if (a.W <= 1024 * NR) {
    if ((a.W & 3) == 0) affine_seam_row<true, NR>(a, t, s44); else affine_seam_row<false, NR>(a, t, s44);
    return;
  }
  if constexpr (NR < ROW_REG) return;
  float* s4 = s44[0];
  float* xt = a.x + t * a.W;
  float* yt = a.ytmp + t * a.W;
  for (int c = threadIdx.x; c < a.W; c += 256) {
    float v = 0.f;
    for (int k = 0; k < a.top; k++) v += a.y[(t * a.top + k) * a.W + c];
    if (a.ysh) v += a.ysh[t * a.W + c];
    yt[c] = v;
  }
  float mean, rstd;
  row_moments_256(yt, a.W, a.eps, s4, mean, rstd);      // (a thread reads back only what it wrote)
  for (int c = threadIdx.x; c < a.W; c += 256) xt[c] = fmaf(a.mult, fmaf((yt[c] - mean) * rstd, a.w_post[c], a.b_post[c]), xt[c]);
  if (!a.w_next) return;
  row_moments_256(xt, a.W, a.eps, s4, mean, rstd);
  for (int c = threadIdx.x; c < a.W; c += 256) a.out[t * a.W + c] = fmaf((xt[c] - mean) * rstd, a.w_next[c], a.b_next[c]);
}
template <int NR>
__global__ __launch_bounds__(256) void affine_seam_kernel(AffineSeamArgs a) { affine_seam_body<NR>(a); }
template <int NR>
__global__ __launch_bounds__(256) void affine_seam_route_kernel(AffineSeamArgs a, RouterGroupArgs r) {      // (as sandwich_route_kernel)
  const RouterAhead ahead = router_ahead(r.in, r.corr, r.E);
  affine_seam_body<NR>(a);
  __syncthreads();
  router_group_lanes(r, ahead);
}

// ---- sigmoid attention with mixed heads.  For the query token i and every key j it sees (a sliding window, a chunk, or all before it: stack_meta.h):
//   w_g(i, j) = sigmoid(q_g(i) . k_kv(g)(j) * scale + pb[g])          per query head g, not normalised over the keys
//   w'_h(i, j) = sum_g talk[h][g] w_g(i, j)                            the heads' weights mixed (talk nullptr: w' = w)
//   out_h(i) = sum_j w'_h(i, j) v_kv(h)(j)                             head h keeps its own key / value head
// and out_h is multiplied by sigmoid(gate) per channel where a gate is given.  Every key, also those of the step's own tokens, is read from the pool.
// One workgroup per token (and per share of its keys in the split form).  Keys are taken KT at a time:
//   scores   the tile's (key, head) pairs are dealt to the threads: a key row against the head's query (queries in LDS, read as broadcasts), sigmoid
//   mix      the pairs again: a pair's mixed weight from its key's `heads` weights in LDS
//   values   a thread owns NPT output channels (head, c), or NPT slices of eight channels where rows are 16-byte aligned (VEC): it walks the tile's keys,
//            reading weights from LDS and value rows coalesced from the pool
// Nothing is normalised, so the shares of a divided window are simply added (sigmoid_mix_merge_kernel, in split order).
struct MixAttnArgs {
  const float* q; long long ldq;        // head h of token t at q + t * ldq + h * dim
  const void* poolK; const void* poolV; // [pages][page_tokens][kv_heads * dim], [pages][page_tokens][kv_heads * vdim]
  const float* pb;                      // [heads] (nullptr: no bias)
  const float* talk;                    // [heads][heads] (nullptr: heads are not mixed)
  const float* gate; long long ldg;     // gate pre-activation of (t, h, c) at gate + t * ldg + h * vdim + c (nullptr: none)
  float* out; long long ldo;            // [T][heads * vdim]
  int heads, kv_heads, dim, vdim, kt;   // kt: keys per tile (<= 256)
  float scale;
  int mask_kind, mask_size;
  float* part; int nsplit, keys_per;    // split form: part [T][nsplit][heads * vdim]; split z takes keys_per keys from the first visible key on
  // sigmoid_mix_step_kernel, single tokens: q holds the projections' row [q | k | v] as it comes, and the step appends the token itself (gqa_append_kernel's part): heads of q and k
  // divided by sqrt(mean(head^2) + unit_eps) where that is positive, the row stored; poolVT: the values' transposed copy (nullptr: none)
  int append; float unit_eps; void* poolVT;
};
inline size_t mix_attn_lds_bytes(int heads, int dim, int kt) { return ((size_t)heads * dim + 2 * (size_t)heads * kt + (size_t)heads * heads) * 4 + (size_t)kt * 4; }
template <int DT, int NPT, bool VEC, bool SPLIT>
__global__ __launch_bounds__(256) void sigmoid_mix_attn_kernel(StepMeta m, MixAttnArgs a) {
  extern __shared__ __attribute__((aligned(16))) float s_mix[];
  const int H = a.heads, G = a.kv_heads, qpg = H / G, KT = a.kt, tid = threadIdx.x;
  float* s_q = s_mix;                        // [H][dim]
  float* s_w = s_q + (size_t)H * a.dim;      // [H][KT] sigmoid weights
  float* s_w2 = s_w + (size_t)H * KT;        // [H][KT] mixed weights
  float* s_t = s_w2 + (size_t)H * KT;        // [H][H]
  int* s_slot = reinterpret_cast<int*>(s_t + (size_t)H * H);      // [KT] pool row of the tile's keys
  const int t = blockIdx.x, row = m.tok_row[t], pos = m.tok_pos[t];
  int k0 = first_key(pos, a.mask_kind, a.mask_size), k1 = pos + 1;
  if (SPLIT) { k0 = min(k1, k0 + (int)blockIdx.y * a.keys_per); k1 = min(k1, k0 + a.keys_per); }
  const float* q = a.q + (size_t)t * a.ldq;
  for (int i = tid; i < H * a.dim; i += 256) s_q[i] = q[i];
  if (a.talk) for (int i = tid; i < H * H; i += 256) s_t[i] = a.talk[i];
  const int kd = G * a.dim, vd = G * a.vdim, O = H * a.vdim, pmask = (1 << m.page_shift) - 1;
  const elem_t<DT>* pk = reinterpret_cast<const elem_t<DT>*>(a.poolK);
  const elem_t<DT>* pv = reinterpret_cast<const elem_t<DT>*>(a.poolV);
  // a thread's outputs: NPT channels (tid + 256 n), or with VEC NPT slices of eight neighbouring channels of one head (slice tid + 256 n)
  constexpr int CW = VEC ? 8 : 1;
  float acc[NPT][CW];
  int oh[NPT], ov[NPT];      // the output's head and its (first) column in a value row
#pragma unroll
  for (int n = 0; n < NPT; n++) {
    const int o = (tid + 256 * n) * CW, h = o < O ? o / a.vdim : 0;
#pragma unroll
    for (int e = 0; e < CW; e++) acc[n][e] = 0.f;
    oh[n] = h; ov[n] = (h / qpg) * a.vdim + (o < O ? o - h * a.vdim : 0);
  }
  for (int kb = k0; kb < k1; kb += KT) {
    const int nk = min(KT, k1 - kb);
    __syncthreads();                         // queries staged; the previous tile's weights and rows have been read
    if (tid < nk) {
      const int j = kb + tid;
      const int page = m.tbl[(size_t)row * m.tbl_stride + (j >> m.page_shift)];
      s_slot[tid] = (page << m.page_shift) + (j & pmask);
    }
    __syncthreads();
    for (int i = tid; i < nk * H; i += 256) {      // scores: one (key, head) pair per thread and round; neighbours take neighbouring keys of one head
      const int g = i / nk, jj = i - g * nk;
      const elem_t<DT>* kc = pk + (size_t)s_slot[jj] * kd + (size_t)(g / qpg) * a.dim;
      const float* qg = s_q + (size_t)g * a.dim;
      float s = 0.f;
      if (VEC) {
#pragma unroll 4
        for (int d = 0; d < a.dim; d += 8) {      // (several slices in flight: a step of few tokens is bound by the latency of these loads)
          float f[8];
          slice_unpack<DT>(load_slice<DT>(kc, (size_t)(d >> 3)), f);
          const f32x4 qa = *reinterpret_cast<const f32x4*>(qg + d), qb = *reinterpret_cast<const f32x4*>(qg + d + 4);
#pragma unroll
          for (int e = 0; e < 4; e++) s = fmaf(qa[e], f[e], s);
#pragma unroll
          for (int e = 0; e < 4; e++) s = fmaf(qb[e], f[4 + e], s);
        }
      } else {
        for (int d = 0; d < a.dim; d++) s = fmaf(qg[d], elem_to_f32<DT>(kc[d]), s);
      }
      s = fmaf(s, a.scale, a.pb ? a.pb[g] : 0.f);
      s_w[(size_t)g * KT + jj] = 1.0f / (1.0f + expf(-s));
    }
    __syncthreads();
    if (a.talk) {
      for (int i = tid; i < nk * H; i += 256) {    // mix: every (key, head) pair reads its key's weights of all heads
        const int h = i / nk, jj = i - h * nk;
        float v = 0.f;
        for (int g = 0; g < H; g++) v = fmaf(s_t[h * H + g], s_w[(size_t)g * KT + jj], v);
        s_w2[(size_t)h * KT + jj] = v;
      }
      __syncthreads();
    }
    const float* sw = a.talk ? s_w2 : s_w;
#pragma unroll 4
    for (int jj = 0; jj < nk; jj++) {
      const elem_t<DT>* vr = pv + (size_t)s_slot[jj] * vd;
#pragma unroll
      for (int n = 0; n < NPT; n++) {
        if ((tid + 256 * n) * CW >= O) continue;
        const float wt = sw[(size_t)oh[n] * KT + jj];
        if constexpr (VEC) {
          float f[8];
          slice_unpack<DT>(load_slice<DT>(vr + ov[n], 0), f);
#pragma unroll
          for (int e = 0; e < 8; e++) acc[n][e] = fmaf(wt, f[e], acc[n][e]);
        } else acc[n][0] = fmaf(wt, elem_to_f32<DT>(vr[ov[n]]), acc[n][0]);
      }
    }
  }
#pragma unroll
  for (int n = 0; n < NPT; n++)
#pragma unroll
    for (int e = 0; e < CW; e++) {
      const int o = (tid + 256 * n) * CW + e;
      if (o >= O) continue;
      if (SPLIT) a.part[((size_t)t * a.nsplit + blockIdx.y) * O + o] = acc[n][e];
      else a.out[(size_t)t * a.ldo + o] = a.gate ? acc[n][e] / (1.0f + expf(-a.gate[(size_t)t * a.ldg + o])) : acc[n][e];
    }
}
// The split form of few tokens, whose workgroups each have a tile or two: bound by the chain of their loads (a key row a thread, four slices of it on their way, then the tile's value
// rows four at a time: 18.5 us for two tokens over 1024 keys, 64 workgroups).  Here every load of a tile of 32 keys stands at once in whole lines: four keys a wave and turn, sixteen
// lanes a key row, for the scores; a slice of eight value channels and every KG-th key a thread for the values, whose key groups meet in LDS.  9.0 us for the same (14.2 with runtime divisions in its index arithmetic and a sigmoid per head and lane).
// Where every token is alone in its entry it also appends: 10.1 us in one launch where the walk was 9.1 and the append 5.3.
// Rows of 16-byte slices, dim <= 128, at most 16 heads of at most four a key / value head, at most 256 value slices (mix_step_ok), rows of q at 16 bytes.
constexpr int MIX_STEP_HEADS = 16, MIX_STEP_GROUP = 4, MIX_STEP_KEYS = 32;
inline bool mix_step_ok(int heads, int kv_heads, int dim, int vdim) {
  return dim % 8 == 0 && dim <= 128 && vdim % 8 == 0 && heads <= MIX_STEP_HEADS && heads <= MIX_STEP_GROUP * kv_heads && kv_heads * vdim <= 2048;
}
template <int DT>
__global__ __launch_bounds__(256) void sigmoid_mix_step_kernel(StepMeta m, MixAttnArgs a) {
  constexpr int KT = MIX_STEP_KEYS, MQ = MIX_STEP_GROUP;
  __shared__ __attribute__((aligned(16))) float s_q[MIX_STEP_HEADS][128];
  __shared__ float s_w[MIX_STEP_HEADS][KT + 1], s_w2[MIX_STEP_HEADS][KT + 1], s_t[MIX_STEP_HEADS][MIX_STEP_HEADS], s_acc[MQ * 8][256];
  const int H = a.heads, G = a.kv_heads, qpg = H / G, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, sub = lane >> 4, ch = 8 * (lane & 15);
  const int t = blockIdx.x, row = m.tok_row[t], pos = m.tok_pos[t], pmask = (1 << m.page_shift) - 1, kd = G * a.dim, vd = G * a.vdim;
  int k1 = pos + 1;
  const int k0 = min(k1, first_key(pos, a.mask_kind, a.mask_size) + (int)blockIdx.y * a.keys_per);
  k1 = min(k1, k0 + a.keys_per);
  const int* tbl = m.tbl + (size_t)row * m.tbl_stride;
  auto slot_of = [&](int key) -> size_t { return ((size_t)tbl[key >> m.page_shift] << m.page_shift) + (size_t)(key & pmask); };
  const elem_t<DT>* pk = reinterpret_cast<const elem_t<DT>*>(a.poolK);
  const elem_t<DT>* pv = reinterpret_cast<const elem_t<DT>*>(a.poolV);
  const int slices = vd >> 3, KG = 256 / slices, kg = tid / slices, sl = tid - kg * slices, vg = sl / (a.vdim >> 3);      // key groups; this thread's group, slice and key / value head
  auto head = [&](const float* r) -> f32x4 {      // this lane's four channels of a head's 32, as the attention takes them
    const int c = 4 * (tid & 31);
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    if (c < a.dim) x = *reinterpret_cast<const f32x4*>(r + c);
    if (a.append && a.unit_eps > 0.f) {
      const float ss = row_group_sum<32>(fmaf(x[0], x[0], x[1] * x[1]) + fmaf(x[2], x[2], x[3] * x[3]));
      x *= 1.0f / sqrtf(ss / (float)a.dim + a.unit_eps);
    }
    return x;
  };
  const float* qr = a.q + (size_t)t * a.ldq;
  if (a.append && k1 == pos + 1 && k0 < k1) {      // (uniform) the share that ends with the token's own key stores its row before any of its keys is read
    const float *kr = qr + (size_t)H * a.dim, *vr = kr + kd;
    elem_t<DT>*kdst = reinterpret_cast<elem_t<DT>*>(const_cast<void*>(a.poolK)) + slot_of(pos) * kd, *vdst = reinterpret_cast<elem_t<DT>*>(const_cast<void*>(a.poolV)) + slot_of(pos) * vd;
    for (int g = tid >> 5; g < G; g += 8) {
      const f32x4 x = head(kr + (size_t)g * a.dim);
      if (4 * (tid & 31) < a.dim)
#pragma unroll
        for (int e = 0; e < 4; e++) kdst[(size_t)g * a.dim + 4 * (tid & 31) + e] = f32_to_elem<DT>(x[e]);
    }
    elem_t<DT>* vt = a.poolVT ? reinterpret_cast<elem_t<DT>*>(a.poolVT) + (((size_t)tbl[pos >> m.page_shift] * vd) << m.page_shift) + (size_t)(pos & pmask) : nullptr;
    for (int c = tid; c < vd; c += 256) {
      const elem_t<DT> e = f32_to_elem<DT>(vr[c]);
      vdst[c] = e;
      if (vt) vt[(size_t)c << m.page_shift] = e;
    }
    __threadfence_block();
    __syncthreads();
  }
  for (int h = tid >> 5; h < H; h += 8) {
    const f32x4 x = head(qr + (size_t)h * a.dim);
    if (4 * (tid & 31) < a.dim) *reinterpret_cast<f32x4*>(&s_q[h][4 * (tid & 31)]) = x;
  }
  if (a.talk && (tid >> 4) < H && (tid & 15) < H) s_t[tid >> 4][tid & 15] = a.talk[(tid >> 4) * H + (tid & 15)];
  float acc[MQ][8];
#pragma unroll
  for (int r = 0; r < MQ; r++)
#pragma unroll
    for (int e = 0; e < 8; e++) acc[r][e] = 0.f;
  for (int kb = k0; kb < k1; kb += KT) {
    const int last = k1 - 1, nk = min(KT, k1 - kb);
    Slice8<DT> vr[4];
    auto values = [&](int i0) {
#pragma unroll
      for (int u = 0; u < 4; u++) vr[u] = load_slice<DT>(pv + slot_of(min(kb + i0 + u * KG, last)) * vd + 8 * sl, 0);
    };
    if (kg < KG) values(kg);
    __syncthreads();                         // queries staged; the previous tile's weights have been read
    for (int g0 = 0; g0 < G; g0 += 2) {
      Slice8<DT> kr[2][2];
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const elem_t<DT>* kp = pk + slot_of(min(kb + 4 * (wv + 4 * u) + sub, last)) * kd + min(ch, a.dim - 8);
#pragma unroll
        for (int x = 0; x < 2; x++) kr[u][x] = load_slice<DT>(kp + min(g0 + x, G - 1) * a.dim, 0);
      }
#pragma unroll
      for (int u = 0; u < 2; u++)
#pragma unroll
        for (int x = 0; x < 2; x++) {
          const int g = g0 + x, i = 4 * (wv + 4 * u) + sub;
          if (g >= G) continue;
          float k[8], sc[MQ] = {0.f, 0.f, 0.f, 0.f};
          slice_unpack<DT>(kr[u][x], k);
          if (ch < a.dim)
#pragma unroll
            for (int r = 0; r < MQ; r++) {
              const float* q = s_q[min(g * qpg + r, H - 1)] + ch;
              const f32x4 qa = *reinterpret_cast<const f32x4*>(q), qb = *reinterpret_cast<const f32x4*>(q + 4);
#pragma unroll
              for (int e = 0; e < 8; e++) sc[r] = fmaf(e < 4 ? qa[e & 3] : qb[e & 3], k[e], sc[r]);
            }
          float v = 0.f;                     // lane r of a key's sixteen keeps head r
#pragma unroll
          for (int r = 0; r < MQ; r++) { const float z = row_group_sum<16>(sc[r]); v = (lane & 15) == r ? z : v; }
          const int h = min(g * qpg + (lane & 15), H - 1);
          v = 1.0f / (1.0f + expf(-fmaf(v, a.scale, a.pb ? a.pb[h] : 0.f)));
          if ((lane & 15) < qpg) s_w[h][i] = v;
        }
    }
    __syncthreads();
    if (a.talk) {
      for (int h = tid / KT; h < H; h += 256 / KT) {
        const int j = tid % KT;
        float v = 0.f;
#pragma unroll 4
        for (int g = 0; g < H; g++) v = fmaf(s_t[h][g], s_w[g][j], v);
        s_w2[h][j] = v;
      }
      __syncthreads();
    }
    auto weight = [&](int h, int j) { return a.talk ? s_w2[h][j] : s_w[h][j]; };
    if (kg < KG)
      for (int i0 = kg; i0 < nk; i0 += 4 * KG) {
        if (i0 != kg) values(i0);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int i = i0 + u * KG;
          if (i >= nk) continue;
          float f[8];
          slice_unpack<DT>(vr[u], f);
#pragma unroll
          for (int r = 0; r < MQ; r++) {
            const float w = weight(min(vg * qpg + r, H - 1), i);
#pragma unroll
            for (int e = 0; e < 8; e++) acc[r][e] = fmaf(w, f[e], acc[r][e]);
          }
        }
      }
  }
#pragma unroll
  for (int r = 0; r < MQ; r++)
#pragma unroll
    for (int e = 0; e < 8; e++) s_acc[r * 8 + e][tid] = acc[r][e];
  __syncthreads();
  float* part = a.part + ((size_t)t * a.nsplit + blockIdx.y) * H * a.vdim;
  for (int c = tid; c < vd; c += 256) {      // a channel of a value row, for every head that reads it
    const int g = c / a.vdim;
    float v[MQ] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = 0; k < KG; k++)
#pragma unroll
      for (int r = 0; r < MQ; r++) v[r] += s_acc[r * 8 + (c & 7)][k * slices + (c >> 3)];
#pragma unroll
    for (int r = 0; r < MQ; r++) if (r < qpg) part[(size_t)(g * qpg + r) * a.vdim + c - g * a.vdim] = v[r];
  }
}
__global__ __launch_bounds__(256) void sigmoid_mix_merge_kernel(MixAttnArgs a) {
  const size_t t = blockIdx.x;
  const int O = a.heads * a.vdim;
  for (int o = threadIdx.x + 256 * blockIdx.y; o < O; o += 256 * gridDim.y) {
    float v = 0.f;
#pragma unroll 8
    for (int s = 0; s < a.nsplit; s++) v += a.part[(t * a.nsplit + s) * O + o];
    a.out[t * a.ldo + o] = a.gate ? v / (1.0f + expf(-a.gate[t * a.ldg + o])) : v;
  }
}

}  // namespace tgx
