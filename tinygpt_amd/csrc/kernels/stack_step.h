// stack_step.h — one decoded token of a mixer in ONE launch: what stands between the mixer's products.  First the recurrences, then attention over a short context.  A step of single tokens is bound by its launches (2.4 us for an
// empty one), and a recurrence took three to five of them: the low-rank decay's second product or the convolution with its norms and gates, the rotation, the scan, the norm and gate
// behind it.  Here a workgroup owns a head of one entry with all of its value columns, so that nothing crosses workgroups: the head's inputs are made in LDS, the state [dim][vdim]
// passes through the registers of 1024 threads once (rows of it are read and written whole, 256 bytes a wave and row; the scan's workgroups of sixteen columns take 64-byte
// pieces) and is on its way before anything else is computed, and the outputs are normed and gated where they are.
// The arithmetic is that of the kernels it stands for (stack_rec.h, stack_seq.h), fp32 throughout; sums over the key channels and over a head's outputs meet in another order.
//
// Threads: column j = tid & (CP - 1) (CP: vdim rounded up to a power of two), row group tid / CP with DPER rows each.
// Measured, us a launch in a decoded step's trace (the launches that it stands for): one stream, wkv of 16 heads of 64 x 64 with its decays 5.2 (3.8, 4.1, 2.5); sixteen entries, channel
// decays of 8 heads of 128 x 128 8.8 (convolution 5.4, scan 11.7, norm 3.3), retention of 4 heads of 128 x 256 with its rotation 8.8 (3.7, 9.3, 3.0).
// What bounds it is latency: the launch, the step's tables, the loads that depend on them, three meetings of the waves.  So no load waits for another that it does not depend on: all of them, the state last,
// are asked for before anything is computed, with clamped places in place of branches.  A convolution's taps one after the other, four slices of a decay's product, and conditional loads, whose registers
// the compiler waits for where branches meet, were up to ten round trips: channel decays 9.2 -> 8.9, retention 9.4 -> 8.8, a delta rule beside attention 8.9 -> 7.9 (with attention as below).  Eight waves
// with twice the rows each are no faster (9.6, 8.7; retention's rows do not fit them).
#pragma once
#include "stack_rec.h"
#include "stack_seq.h"

namespace tgx {

constexpr int STEP_MAX_DIM = 256, STEP_MAX_TAPS = 8, STEP_THREADS = 1024;
struct RecStepArgs {
  RecScanArgs s;             // the recurrence (rec_scan_kernel); with prep its a, k, v, beta and g are made here instead
  DeltaPrepArgs p; int prep; // the convolved inputs (delta_prep_kernel)
  const float* cs; int rot_dims;      // q and k turn first (gqa_append_kernel, halves): [position][rot_dims / 2][2]; nullptr: not
  const void* w2; const float* lora; const float* w0; int rank, terms;      // wkv: the decays as exp(-exp(w0 + W2 lora)), W2 [heads * dim][rank] in the storage type (nullptr: given in s.w)
  long long ldlora;
  HeadNormGateArgs g;        // the norm and gate behind the head (its hs is not read)
};

template <int DT, int KIND, int DPER>
__device__ __forceinline__ void rec_step_body(const StepMeta& m, const RecStepArgs& a, const int log_cp, const int e, const int h) {
  constexpr int NT = STEP_THREADS;
  __shared__ __attribute__((aligned(16))) float s_q[STEP_MAX_DIM + 8], s_k[STEP_MAX_DIM + 8], s_w[STEP_MAX_DIM + 8];      // (zeros behind dim)
  __shared__ float s_v[STEP_MAX_DIM], s_b[2], s_n[16], s_unit[2];
  __shared__ float s_pk[NT], s_po[NT];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int t = e, row = m.tok_row[t], pos = m.tok_pos[t], par = m.tok_par[t];      // (an entry is a token)
  const int dim = a.s.dim, vdim = a.s.vdim, share = a.s.heads / a.s.kv_heads, kh = h / share;
  const int cp = 1 << log_cp, RG = NT >> log_cp, j = tid & (cp - 1), rg = tid >> log_cp, d0 = rg * DPER;
  const bool col = j < vdim;
  // What a thread needs beside the state is asked for here, all of it, in front of the state: the first slices of a wkv head's decay product (sixteen lanes a channel, four elements a lane), the
  // output's gate and norm weight.  (A slice after the other they were four round trips.)
  // A convolution in front of 32 rows a lane has no registers for that (they spilled: 256 x 128, sixteen entries 15.6 us, 13.7 so): there everything is asked for where it is used.
  constexpr bool PREP = KIND == REC_DELTA || KIND == REC_CDELTA, AHEAD = !PREP || DPER <= 16;
  const bool mine = tid < vdim;
  float gate = 0.f, w_out = 1.f;
  auto out_operands = [&] {
    const int out_c = min(tid, vdim - 1);
    const float* gp = a.g.gate + (size_t)t * a.g.ldg + (size_t)h * vdim;
    gate = gp[out_c]; w_out = (a.g.w ? a.g.w + (size_t)h * a.g.w_hstride : gp)[out_c];
  };
  if (AHEAD) out_operands();
  constexpr bool W2 = KIND == REC_WKV;
  typename std::conditional<DT == DT_F32, float, unsigned>::type w2r[W2 ? 4 : 1];      // (as they lie in memory: widened where they are used)
  float lor[W2 ? 4 : 1], w0 = 0.f;
  auto decay_slices = [&](int c0, int r0) {
    const size_t at = (size_t)h * dim + min(c0 + (tid >> 4), dim - 1);
#pragma unroll
    for (int i = 0; i < (W2 ? 4 : 0); i++) { const int k = min(r0 + (tid & 15) + 16 * i, a.rank - 1); w2r[i] = reinterpret_cast<const elem_t<DT>*>(a.w2)[at * a.rank + k]; lor[i] = a.lora[(size_t)t * a.ldlora + k]; }
    if (r0 == 0) w0 = a.w0[at];
  };
  if (W2 && a.w2) decay_slices(0, 0);
  // ... and the raw row, taps and tails of a convolved channel, in the waves that have any: taps that the filter has not and channels again in idle waves were 15 loads a thread more than
  // their data, in line with the state's (8 heads of 128 x 128, one / four / sixteen entries: delta rule 7.9 / 8.5 / 9.5 us, so 7.1 / 7.6 / 8.8)
  const DeltaPrepArgs& p = a.p;
  const int GD = p.kv_heads * dim, C = 2 * GD + p.heads * vdim, nb = p.taps - 1, ct = min(tid, 2 * dim + vdim - 1), part = ct < dim ? 0 : ct < 2 * dim ? 1 : 2, cc = ct - part * dim;
  const int c = part == 0 ? kh * dim + cc : part == 1 ? GD + kh * dim + cc : 2 * GD + h * vdim + cc;
  const size_t tail = (size_t)row * nb * C + c;
  float zb = 0.f, za_raw = 0.f, za_bias = 0.f, al = 0.f;
  auto gates = [&] {
    const float* pr = p.proj + (size_t)t * p.ldp + p.col0 + p.b_col + h;
    zb = pr[0];
    if (p.a_log) { za_raw = pr[p.heads]; za_bias = p.dt_bias[h]; al = p.a_log[h]; }
  };
  float x0 = 0.f, cw[PREP ? STEP_MAX_TAPS : 1], old[PREP ? STEP_MAX_TAPS : 1];      // old[d]: the row d positions back
  auto channel = [&] {
    x0 = p.proj[(size_t)t * p.ldp + p.col0 + c];
#pragma unroll
    for (int d = 0; d < (PREP ? STEP_MAX_TAPS : 0); d++) if (d <= nb) cw[d] = p.cw[(size_t)c * p.taps + nb - d];
#pragma unroll
    for (int d = 1; d < (PREP ? STEP_MAX_TAPS : 0); d++) if (d <= nb) old[d] = p.state[(size_t)par * p.state_buf + tail + (size_t)(nb - d) * C];
  };
  if (PREP && AHEAD && a.prep) {
    gates();
    if (64 * __builtin_amdgcn_readfirstlane(wv) < 2 * dim + vdim) channel();
  }
  float* Sg = a.s.S + ((size_t)row * a.s.heads + h) * (size_t)dim * vdim;
  float S[DPER], ub[KIND == REC_WKV ? DPER : 1];
#pragma unroll
  for (int dd = 0; dd < DPER; dd++) {
    const int d = d0 + dd;
    if (AHEAD) S[dd] = Sg[(size_t)min(d, dim - 1) * vdim + min(j, vdim - 1)];      // (rows and columns that are not there: below)
    else S[dd] = (pos != 0 && d < dim && col) ? Sg[(size_t)d * vdim + j] : 0.f;
    if (KIND == REC_WKV) ub[dd] = a.s.u[(size_t)h * dim + min(d, dim - 1)];
  }
  // ---- the head's inputs
  if (tid < 8) s_q[dim + tid] = s_k[dim + tid] = s_w[dim + tid] = 0.f;
  if (PREP && a.prep) {
    if (tid < 2 * dim + vdim) {
      if (!AHEAD) channel();
      float acc = cw[0] * x0;
#pragma unroll
      for (int d = 1; d < (PREP ? STEP_MAX_TAPS : 0); d++) {
        if (d > nb) continue;
        if (pos - d < 0) old[d] = 0.f;
        acc = fmaf(cw[d], old[d], acc);
      }
      const float act = acc / (1.0f + expf(-acc));
      if (part == 0) s_q[cc] = act; else if (part == 1) s_k[cc] = act; else s_v[cc] = act;
      if (nb > 0 && (part == 2 || h == kh * share)) {              // (heads that share keys: the first of them moves the tails)
        float* st_new = p.state + (size_t)(par ^ 1) * p.state_buf + tail;
        st_new[(size_t)(nb - 1) * C] = x0;
#pragma unroll
        for (int d = 1; d < (PREP ? STEP_MAX_TAPS : 0) - 1; d++) if (d < nb) st_new[(size_t)(nb - 1 - d) * C] = old[d];
      }
    }
    if (tid == NT - 1) {
      if (!AHEAD) gates();
      const float za = za_raw + za_bias;
      s_b[0] = 1.0f / (1.0f + expf(-zb));
      if (p.a_log) {
        const float sp = za > 20.f ? za : log1pf(expf(za));
        s_b[1] = expf(-expf(al) * sp);
      }
    }
    if (KIND == REC_CDELTA && tid < dim) s_w[tid] = a.s.w[(size_t)t * a.s.ldw + (size_t)h * dim + tid];
    __syncthreads();
    if (wv < 2) {                                                  // the norms of q and k
      const float* u = wv ? s_k : s_q;
      float ss = 0.f;
      for (int c = lane; c < dim; c += 64) ss = fmaf(u[c], u[c], ss);
      ss = wave_sum(ss);
      if (lane == 0) s_unit[wv] = (wv ? 1.0f : p.q_scale) / sqrtf(ss + p.unit_eps);
    }
    __syncthreads();
  } else {
    if (tid < dim) {
      const float* q = a.s.a + (size_t)t * a.s.lda + (size_t)kh * dim;
      const float* k = a.s.k + (size_t)t * a.s.ldk + (size_t)kh * dim;
      float qv = q[tid], kv = k[tid];
      const int half = a.cs ? a.rot_dims >> 1 : 0;
      if (tid < 2 * half) {
        const int at = tid < half ? tid : tid - half, other = tid < half ? tid + half : at;
        const float c = a.cs[((size_t)pos * half + at) * 2], s = a.cs[((size_t)pos * half + at) * 2 + 1], q1 = q[other], k1 = k[other];
        qv = tid < half ? __fsub_rn(__fmul_rn(qv, c), __fmul_rn(q1, s)) : __fadd_rn(__fmul_rn(qv, c), __fmul_rn(q1, s));
        kv = tid < half ? __fsub_rn(__fmul_rn(kv, c), __fmul_rn(k1, s)) : __fadd_rn(__fmul_rn(kv, c), __fmul_rn(k1, s));
      }
      s_q[tid] = qv; s_k[tid] = kv;
      if ((KIND == REC_CDELTA || KIND == REC_WKV) && !a.w2) s_w[tid] = a.s.w[(size_t)t * a.s.ldw + (size_t)(KIND == REC_WKV ? kh : h) * dim + tid];
    }
    if (tid >= NT - vdim) s_v[tid - (NT - vdim)] = a.s.v[(size_t)t * a.s.ldv + (size_t)h * vdim + tid - (NT - vdim)];      // (in other threads than q and k where there are enough)
    if (KIND != REC_WKV && tid == NT - 1) {
      const size_t at = (size_t)t * a.s.ldg + h;
      if (KIND == REC_SSD && a.s.fixed) { s_b[0] = a.s.beta0; s_b[1] = a.s.fixed[h]; }
      else { s_b[0] = a.s.beta[at]; if (KIND != REC_CDELTA) s_b[1] = a.s.g[at]; }
    }
    if (W2 && a.w2) {
      for (int c0 = 0; c0 < dim; c0 += NT / 16) {
        const int c = c0 + (tid >> 4);
        float acc = 0.f;
        for (int r0 = 0; r0 < a.rank; r0 += 64) {
          if (c0 + r0 > 0) decay_slices(c0, r0);
#pragma unroll
          for (int i = 0; i < (W2 ? 4 : 0); i++)
            if (r0 + (tid & 15) + 16 * i < a.rank) acc = fmaf(elem_to_f32<DT>((elem_t<DT>)w2r[i]), round_storage_if<DT>(lor[i], a.terms == 1), acc);
        }
        acc = row_group_sum<16>(acc);
        if ((tid & 15) == 0 && c < dim) s_w[c] = expf(-expf(acc + w0));
      }
    }
    if (tid < 2) s_unit[tid] = 1.f;
    __syncthreads();
  }
  // ---- the recurrence.  (A wave's lanes stand at one row group, so the inputs' reads are broadcasts; the unit norms of q and k multiply the sums.)
  const float vj = col ? s_v[j] : 0.f, uq = s_unit[0], uk = s_unit[1];
  auto of = [&](const float* p, int dd) { return *reinterpret_cast<const f32x4*>(p + min(d0 + dd, (dim + 3) & ~3)); };      // (rows past dim: zeros)
  auto total = [&](const float* p) {                               // a column's row groups, four on their way at a time
    float x = 0.f;
    for (int r = 0; r < RG; r += 4) {
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; i++) y[i] = p[((r + i) << log_cp) + j];
      x += (y[0] + y[1]) + (y[2] + y[3]);
    }
    return x;
  };
  float po = 0.f;
#pragma unroll
  for (int dd = 0; dd < DPER; dd++) {
    if (AHEAD && (pos == 0 || d0 + dd >= dim || !col)) S[dd] = 0.f;
    if (KIND == REC_WKV && d0 + dd >= dim) ub[dd] = 0.f;
  }
  if (KIND == REC_WKV) {
#pragma unroll
    for (int dd = 0; dd < DPER; dd += 4) {
      const f32x4 q = of(s_q, dd), k = of(s_k, dd), w = of(s_w, dd);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float kv = k[i] * vj;
        po = fmaf(q[i], fmaf(ub[dd + i], kv, S[dd + i]), po);
        S[dd + i] = fmaf(w[i], S[dd + i], kv);
      }
    }
  } else if (KIND == REC_SSD) {
    const float bv = s_b[0] * vj, g = s_b[1];
#pragma unroll
    for (int dd = 0; dd < DPER; dd += 4) {
      const f32x4 q = of(s_q, dd), k = of(s_k, dd);
#pragma unroll
      for (int i = 0; i < 4; i++) { S[dd + i] = fmaf(g, S[dd + i], k[i] * bv); po = fmaf(S[dd + i], q[i], po); }
    }
  } else {
    float pk = 0.f;
    const float g = KIND == REC_CDELTA ? 1.f : s_b[1];
#pragma unroll
    for (int dd = 0; dd < DPER; dd += 4) {
      const f32x4 k = of(s_k, dd), w = KIND == REC_CDELTA ? of(s_w, dd) : f32x4{g, g, g, g};
#pragma unroll
      for (int i = 0; i < 4; i++) { S[dd + i] *= w[i]; pk = fmaf(S[dd + i], k[i], pk); }
    }
    s_pk[tid] = pk;
    __syncthreads();
    const float uj = s_b[0] * (vj - total(s_pk) * uk) * uk;
#pragma unroll
    for (int dd = 0; dd < DPER; dd += 4) {
      const f32x4 q = of(s_q, dd), k = of(s_k, dd);
#pragma unroll
      for (int i = 0; i < 4; i++) { S[dd + i] = fmaf(k[i], uj, S[dd + i]); po = fmaf(S[dd + i], q[i], po); }
    }
    po *= uq;
  }
  s_po[tid] = po;
#pragma unroll
  for (int dd = 0; dd < DPER; dd++) { const int d = d0 + dd; if (d < dim && col) Sg[(size_t)d * vdim + j] = S[dd]; }
  // the outputs, their norm and gate: one thread a column
  if (!AHEAD) out_operands();
  __syncthreads();
  float o = 0.f;
  if (mine) {
    o = total(s_po);
    if (KIND == REC_SSD && a.s.skip) o = fmaf(a.s.skip[h], vj, o);
  }
  const float ws = wave_sum(o * o);
  if (lane == 0) s_n[wv] = ws;
  __syncthreads();
  if (!mine) return;
  float ss = 0.f;
  for (int i = 0; i < (vdim + 63) >> 6; i++) ss += s_n[i];
  const float rinv = 1.0f / sqrtf(ss / (float)vdim + a.g.eps), sg = 1.0f / (1.0f + expf(-gate));
  a.g.out[(size_t)t * a.g.ldo + (size_t)h * vdim + tid] = o * rinv * (a.g.w ? w_out : 1.f) * (a.g.silu_gate ? gate * sg : sg);
}

template <int DT, int KIND, int DPER>
__global__ __launch_bounds__(STEP_THREADS) void rec_step_kernel(StepMeta m, RecStepArgs a, const int log_cp) { rec_step_body<DT, KIND, DPER>(m, a, log_cp, blockIdx.x, blockIdx.y); }

// ---- attention of single tokens over up to STEP_MAX_KEYS keys, the token's own among them.  The divided form took three launches for this (append, a walk of key tiles by matrix
// instructions, merge), the undivided one two, its walk a chain of 1.3 us a tile on a workgroup per key / value head.  Here a workgroup of eight waves owns an entry and a
// query head (those that share a key / value head read its rows from L2): it finishes the token's queries, key and value in LDS (gqa_append_kernel), the first head of a group stores
// the latter two, then
//   scores   four keys a wave at a time, sixteen lanes a key with eight channels each; every wave's keys are on their way at once
//   softmax  every wave for itself, base 2, as in gqa_attn_mfma_kernel (cap, distance slope, sink, mask)
//   values   a key per wave at a time; the waves' sums meet in LDS
// Queries and probabilities stay fp32 (the matrix forms take them as two 16-bit terms).
// Measured, us: one stream of 50 to 95 keys, eight query heads on two key / value heads of 128 x 128 7.9 (append 3.0, undivided walk 7.9); beside a delta rule in one launch 7.9 (a workgroup of sixteen
// waves a key / value head 8.0 and 8.9).  The group's size does not matter to it: eight or sixteen query heads a key / value head, 50 to 85 keys, one entry 7.4 (append 3.2, walk 7.8 to 9.5), sixteen
// 8.0 (4.2, 10.5 to 12.4), beside a delta rule 7.4 (with the rule's launch 19); 220 to 240 keys 14.8 in one launch and 13.2 to 15.7 in three, beside a delta rule 13.1 and 21.
constexpr int STEP_MAX_KEYS = 256, STEP_MAX_VDIM = 128;
struct GqaStepArgs {
  GqaAppendArgs ap;          // the token's row (maps 1, no q_hi, no qk_unit_eps)
  const float* gate; long long ldg; int gate_per_head;
  float* out; long long ldo; float out_scale;
  float scale, sink; int has_sink;
  int mask_kind, mask_size;
  float softcap; int dist_bias;
  const void *poolK, *poolV; // the pools that are read (those of ap where the layer appends)
};
template <int DT, int NT>
__device__ __forceinline__ void gqa_step_body(const StepMeta& m, const GqaStepArgs& a, const int e, const int h) {
  constexpr int NW = NT / 64, KU = STEP_MAX_KEYS / (4 * NW), VU = STEP_MAX_KEYS / NW;      // turns of a wave over keys (four at a time) and over values
  constexpr float LOG2E = 1.4426950408889634f;
  __shared__ __attribute__((aligned(16))) float s_qr[STEP_MAX_DIM], s_kn[STEP_MAX_DIM];
  __shared__ float s_vn[STEP_MAX_VDIM], s_s[STEP_MAX_KEYS], s_acc[NW][STEP_MAX_VDIM];
  const GqaAppendArgs& ap = a.ap;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = m.tok_row[e], pos = m.tok_pos[e], dim = ap.dim, vdim = ap.vdim, Gq = ap.heads / ap.kv_heads, g = h / Gq;
  const int lo = first_key(pos, a.mask_kind, a.mask_size), n = pos - lo + 1, kd = ap.kv_heads * dim, vd = ap.kv_heads * vdim;
  const int* tbl = m.tbl + (size_t)row * m.tbl_stride;
  const bool fresh_key = ap.poolK != nullptr;                      // (a layer that reads another layer's pool appends nothing: its last key stands there)
  const bool appends = fresh_key && h == g * Gq;                   // (one of a group's workgroups stores the token's key and value; all of them make them)
  const int stored = fresh_key ? n - 1 : n, pmask = (1 << m.page_shift) - 1;
  const float* prow = ap.proj + (size_t)e * ap.ldp;
  // Everything that a thread needs of the token's row is asked for first, then the pages, all of them, then rows, and values as they lie in memory: a page asked for between two rows, or a value
  // widened where it is loaded, waits for every load before it.  Keys: four a wave and turn, sixteen lanes a key; values: a key a wave and turn.
  const int out_c = min(tid, vdim - 1);
  const float gate = a.gate ? a.gate[(size_t)e * a.ldg + (a.gate_per_head ? (size_t)h : (size_t)h * vdim + out_c)] : 0.f;
  const int half = ap.rot_dims >> 1, what = wv >> 1;               // waves 0 and 1: the head's queries, 2 and 3: the key, then the value
  const float* qrow = prow + (what == 0 ? (size_t)h * dim : (size_t)ap.heads * dim + (size_t)g * dim);
  const bool turns = what == 0 || (what == 1 && fresh_key);
  float qv[2] = {0.f, 0.f}, qo[2] = {0.f, 0.f}, qc[2] = {1.f, 1.f}, qs[2] = {0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int c = lane + 64 * (wv & 1) + 128 * i;
    if (!turns || c >= dim) break;
    qv[i] = qrow[c];
    if (c < ap.rot_dims) {
      const int p = ap.rot_pairs ? c >> 1 : c < half ? c : c - half;
      qo[i] = qrow[ap.rot_pairs ? c ^ 1 : c < half ? c + half : c - half];
      qc[i] = ap.cs[((size_t)pos * half + p) * 2]; qs[i] = ap.cs[((size_t)pos * half + p) * 2 + 1];
    }
  }
  const int vc = tid - 256;
  const bool own_v = fresh_key && vc >= 0 && vc < vdim;
  const size_t vat0 = (size_t)e * vd + (size_t)g * vdim + vc;
  float own = own_v ? prow[(size_t)ap.heads * dim + kd + (size_t)g * vdim + vc] : 0.f;
  const float first = own_v && ap.vmode == 2 ? ap.vfirst[vat0] : 0.f, lam = own_v && ap.vmode == 2 ? ap.lam[0] : 0.f;
  const size_t own_page = appends ? (size_t)tbl[pos >> m.page_shift] : 0;
  const int sub = lane >> 4, ch = 8 * (lane & 15);
  const elem_t<DT>* pK = reinterpret_cast<const elem_t<DT>*>(a.poolK) + (size_t)g * dim;
  const elem_t<DT>* pV = reinterpret_cast<const elem_t<DT>*>(a.poolV) + (size_t)g * vdim;
  auto key_of = [&](int i) { return lo + min(i, max(stored - 1, 0)); };
  auto slot_of = [&](int page, int i) -> size_t { return ((size_t)page << m.page_shift) + (size_t)(key_of(i) & pmask); };
  int kat[KU], vat[VU];
#pragma unroll
  for (int u = 0; u < KU; u++) { if (4 * NW * u >= n) break; kat[u] = tbl[key_of(4 * (wv + NW * u) + sub) >> m.page_shift]; }      // (uniform; past the last key: the last one's again)
#pragma unroll
  for (int u = 0; u < VU; u++) { if (NW * u >= n) break; vat[u] = tbl[key_of(wv + NW * u) >> m.page_shift]; }
  __builtin_amdgcn_sched_barrier(0);
  Slice8<DT> kr[KU][2];
#pragma unroll
  for (int u = 0; u < KU; u++) {
    if (4 * NW * u >= n) break;
    const elem_t<DT>* kp = pK + slot_of(kat[u], 4 * (wv + NW * u) + sub) * kd;
#pragma unroll
    for (int c = 0; c < 2; c++) if (128 * c < dim) kr[u][c] = load_slice<DT>(kp + min(ch + 128 * c, dim - 8), 0);
  }
  typename std::conditional<DT == DT_F32, float, unsigned>::type vr[VU][2];      // (a register each: packed in pairs they would be waited for)
#pragma unroll
  for (int u = 0; u < VU; u++) {
    if (NW * u >= n) break;
    const elem_t<DT>* vp = pV + slot_of(vat[u], wv + NW * u) * vd;
    vr[u][0] = vp[min(lane, vdim - 1)];
    if (vdim > 64) vr[u][1] = vp[min(lane + 64, vdim - 1)];
  }
  // the token's queries (score scale and log2 e folded in), key and value
  const bool capped = a.softcap > 0.f;
  const float temp = ap.q_temp_coef != 0.f ? fmaf(ap.q_temp_coef, logf((float)((pos + 1) / ap.q_temp_every) + 1.0f), 1.0f) : 1.0f, qscale = capped ? a.scale : a.scale * LOG2E;
  if (turns) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int c = lane + 64 * (wv & 1) + 128 * i;
      if (c >= dim) break;
      float v = qv[i];
      if (c < ap.rot_dims) {
        const bool first_half = ap.rot_pairs ? (c & 1) == 0 : c < half;
        v = first_half ? __fsub_rn(__fmul_rn(v, qc[i]), __fmul_rn(qo[i], qs[i])) : __fadd_rn(__fmul_rn(v, qc[i]), __fmul_rn(qo[i], qs[i]));
      }
      if (what == 0) s_qr[c] = v * temp * qscale;
      else {
        const elem_t<DT> k = f32_to_elem<DT>(v);
        if (appends) reinterpret_cast<elem_t<DT>*>(ap.poolK)[((own_page << m.page_shift) + (size_t)(pos & pmask)) * kd + (size_t)g * dim + c] = k;
        s_kn[c] = elem_to_f32<DT>(k);
      }
    }
  }
  if (own_v) {
    if (ap.vmode == 1 && appends) ap.vfirst[vat0] = own;
    if (ap.vmode == 2) own = fmaf(lam, first, __fmul_rn(1.0f - lam, own));
    const elem_t<DT> sv = f32_to_elem<DT>(own);
    if (appends) {
      reinterpret_cast<elem_t<DT>*>(ap.poolV)[((own_page << m.page_shift) + (size_t)(pos & pmask)) * vd + (size_t)g * vdim + vc] = sv;
      if (ap.poolVT) reinterpret_cast<elem_t<DT>*>(ap.poolVT)[((own_page * vd + (size_t)g * vdim + vc) << m.page_shift) + (size_t)(pos & pmask)] = sv;
    }
    s_vn[vc] = elem_to_f32<DT>(sv);
  }
  __syncthreads();
  // scores
#pragma unroll
  for (int u = 0; u < KU; u++) {
    if (4 * NW * u >= n) break;
    const int i = 4 * (wv + NW * u) + sub;
    float sc = 0.f;
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if (128 * c >= dim) break;
      const int at = ch + 128 * c;
      float k[8];
      slice_unpack<DT>(kr[u][c], k);
      if (fresh_key && i == n - 1) {
#pragma unroll
        for (int x = 0; x < 8; x++) k[x] = s_kn[min(at + x, dim - 1)];
      }
      if (at < dim) {
        const f32x4 q0 = *reinterpret_cast<const f32x4*>(&s_qr[at]), q1 = *reinterpret_cast<const f32x4*>(&s_qr[at + 4]);
#pragma unroll
        for (int x = 0; x < 8; x++) sc = fmaf(k[x], x < 4 ? q0[x & 3] : q1[x & 3], sc);
      }
    }
    sc = row_group_sum<16>(sc);
    if ((lane & 15) == 0 && i < n) s_s[i] = sc;
  }
  __syncthreads();
  // softmax: every wave for itself, keys lane, lane + 64, ..
  const float slope2 = a.dist_bias ? distance_slope(h, ap.heads) * LOG2E : 0.f;
  float p[STEP_MAX_KEYS / 64], mx = a.has_sink ? a.sink * LOG2E : -INFINITY, l = 0.f;
#pragma unroll
  for (int u = 0; u < STEP_MAX_KEYS / 64; u++) {
    p[u] = -INFINITY;
    if (64 * u >= n) continue;                                     // (uniform)
    const int i = lane + 64 * u;
    float v = i < n ? s_s[i] : -INFINITY;
    if (capped && i < n) v = a.softcap * tanhf(v / a.softcap) * LOG2E;
    p[u] = i < n ? fmaf(-slope2, (float)(n - 1 - i), v) : -INFINITY;
    mx = fmaxf(mx, p[u]);
  }
  mx = group_max<64>(mx);
  const bool dead = mx == -INFINITY;
#pragma unroll
  for (int u = 0; u < STEP_MAX_KEYS / 64; u++) { p[u] = dead ? 0.f : __builtin_amdgcn_exp2f(p[u] - mx); l += p[u]; }
  l = wave_sum(l);
  if (a.has_sink) l += __builtin_amdgcn_exp2f(a.sink * LOG2E - mx);
  // values
  float acc[2] = {0.f, 0.f};
#pragma unroll
  for (int u = 0; u < VU; u++) {
    if (NW * u >= n) break;
    const int i = wv + NW * u;
    if (i >= n) break;                                             // (wave-uniform)
    const float w = __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(p[NW * u / 64]), i & 63));      // (NW divides 64)
    const bool last = fresh_key && i == n - 1;
    acc[0] = fmaf(w, last ? s_vn[min(lane, vdim - 1)] : elem_to_f32<DT>((elem_t<DT>)vr[u][0]), acc[0]);
    if (vdim > 64) acc[1] = fmaf(w, last ? s_vn[min(lane + 64, vdim - 1)] : elem_to_f32<DT>((elem_t<DT>)vr[u][1]), acc[1]);
  }
  s_acc[wv][lane] = acc[0]; s_acc[wv][lane + 64] = acc[1];
  __syncthreads();
  if (tid < vdim) {
    float t[NW];
#pragma unroll
    for (int w = 0; w < NW; w++) t[w] = s_acc[w][tid];
#pragma unroll
    for (int o = NW / 2; o > 0; o >>= 1)
#pragma unroll
      for (int w = 0; w < o; w++) t[w] += t[w + o];
    float v = l > 0.f ? t[0] / l : 0.f;
    if (a.gate) v = v / (1.0f + expf(-gate));
    a.out[(size_t)e * a.ldo + (size_t)h * vdim + tid] = v * a.out_scale;
  }
}
template <int DT>
__global__ __launch_bounds__(512) void gqa_step_kernel(StepMeta m, GqaStepArgs a) { gqa_step_body<DT, 512>(m, a, blockIdx.x, blockIdx.y); }

// The same for steps of more query heads than compute units: a workgroup of sixteen waves takes up to STEP_GROUP query heads of a key / value head, whose rows come once for all of them.  A
// workgroup a query head holds all that a wave loads in registers, so that a compute unit takes one at a time, and the second round costs what the first did.  us, a query head a workgroup /
// this form, 60, 120 and 245 keys: 32 entries of eight heads on two of 128 x 128 (256 heads) 7.6, 10.6, 15.5 / 9.4, 13.4, 20.7, 48 entries 12.3, 17.3, 27.4 / 9.3, 12.7, 20.7; sixteen heads on four of
// 64 x 64, sixteen entries (256) 7.2, 9.3, 14.4 / 8.2, 10.0, 15.4, 24 entries 12.2, 16.1, 25.2 / 8.1, 10.2, 15.8, 64 entries 21.3, 29.5, 48.0 / 8.1, 11.2, 16.6; eight heads on four, 48 entries 12.8, 17.5,
// 28.0 / 10.5, 13.2, 21.4, on one 12.2, 17.0, 27.6 / 8.5, 11.6, 19.4.  With a key / value head a query head there is nothing to share: 48 entries of eight 13.1, 17.7, 29.4 / 17.5, 24.0, 39.9.
constexpr int STEP_GROUP = 4;
template <int DT>
__device__ __forceinline__ void gqa_group_step_body(const StepMeta& m, const GqaStepArgs& a, const int e, const int blk) {
  constexpr int MG = STEP_GROUP, KW = STEP_MAX_KEYS / 16;      // keys of a wave
  constexpr float LOG2E = 1.4426950408889634f;
  __shared__ __attribute__((aligned(16))) float s_qr[MG][STEP_MAX_DIM], s_kn[STEP_MAX_DIM];
  __shared__ float s_vn[STEP_MAX_VDIM], s_s[MG][STEP_MAX_KEYS], s_l[MG], s_acc[16][MG][STEP_MAX_VDIM];
  const GqaAppendArgs& ap = a.ap;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = m.tok_row[e], pos = m.tok_pos[e], dim = ap.dim, vdim = ap.vdim, Gq = ap.heads / ap.kv_heads;
  const int blocks = (Gq + MG - 1) / MG, g = blk / blocks, hb = MG * (blk - g * blocks), h0 = g * Gq + hb, nh = min(MG, Gq - hb);      // its key / value head and its query heads
  const int lo = first_key(pos, a.mask_kind, a.mask_size), n = pos - lo + 1, kd = ap.kv_heads * dim, vd = ap.kv_heads * vdim;
  const int* tbl = m.tbl + (size_t)row * m.tbl_stride;
  const bool fresh_key = ap.poolK != nullptr;                      // (a layer that reads another layer's pool appends nothing: its last key stands there)
  const bool appends = fresh_key && hb == 0;                       // (one of a key / value head's workgroups stores the token's key and value; all of them make them)
  const int stored = fresh_key ? n - 1 : n, pmask = (1 << m.page_shift) - 1;
  const float* prow = ap.proj + (size_t)e * ap.ldp;
  // keys and values of this wave, on their way before anything is computed: four keys a turn, sixteen lanes a key; then a key a turn for the values
  const int sub = lane >> 4, ch = 8 * (lane & 15);
  const elem_t<DT>* pK = reinterpret_cast<const elem_t<DT>*>(a.poolK) + (size_t)g * dim;
  const elem_t<DT>* pV = reinterpret_cast<const elem_t<DT>*>(a.poolV) + (size_t)g * vdim;
  auto slot_of = [&](int i) -> size_t { const int key = lo + min(i, max(stored - 1, 0)); return ((size_t)tbl[key >> m.page_shift] << m.page_shift) + (size_t)(key & pmask); };
  Slice8<DT> kr[KW / 4][2];
#pragma unroll
  for (int u = 0; u < KW / 4; u++) {
    const int i = 4 * (wv + 16 * u) + sub;
    if (64 * u >= n) break;                                        // (uniform)
    const elem_t<DT>* kp = pK + slot_of(i) * kd;
#pragma unroll
    for (int c = 0; c < 2; c++) if (128 * c < dim) kr[u][c] = load_slice<DT>(kp + min(ch + 128 * c, dim - 8), 0);
  }
  float vr[KW][2];
#pragma unroll
  for (int u = 0; u < KW; u++) {
    if (16 * u >= n) break;
    const elem_t<DT>* vp = pV + slot_of(wv + 16 * u) * vd;
#pragma unroll
    for (int c = 0; c < 2; c++) vr[u][c] = 64 * c < vdim ? elem_to_f32<DT>(vp[min(lane + 64 * c, vdim - 1)]) : 0.f;
  }
  // the token's queries (score scale and log2 e folded in), key and value
  const bool capped = a.softcap > 0.f;
  const float temp = ap.q_temp_coef != 0.f ? fmaf(ap.q_temp_coef, logf((float)((pos + 1) / ap.q_temp_every) + 1.0f), 1.0f) : 1.0f, qscale = capped ? a.scale : a.scale * LOG2E;
  const int nq = nh + (fresh_key ? 1 : 0);
  if (wv < 2 * nq)                                                 // two waves a row
    for (int c = lane + 64 * (wv & 1); c < dim; c += 128) {
      const int r = wv >> 1;
      const float* u = prow + (r < nh ? (size_t)(h0 + r) * dim : (size_t)ap.heads * dim + (size_t)g * dim);
      float v = u[c];
      if (c < ap.rot_dims) {
        const int half = ap.rot_dims >> 1, p = ap.rot_pairs ? c >> 1 : c < half ? c : c - half;
        const bool first = ap.rot_pairs ? (c & 1) == 0 : c < half;
        const float cs = ap.cs[((size_t)pos * half + p) * 2], sn = ap.cs[((size_t)pos * half + p) * 2 + 1], o = u[ap.rot_pairs ? c ^ 1 : first ? c + half : c - half];
        v = first ? __fsub_rn(__fmul_rn(v, cs), __fmul_rn(o, sn)) : __fadd_rn(__fmul_rn(v, cs), __fmul_rn(o, sn));
      }
      if (r < nh) s_qr[r][c] = v * temp * qscale;
      else {
        const elem_t<DT> k = f32_to_elem<DT>(v);
        if (appends) reinterpret_cast<elem_t<DT>*>(ap.poolK)[(((size_t)tbl[pos >> m.page_shift] << m.page_shift) + (size_t)(pos & pmask)) * kd + (size_t)g * dim + c] = k;
        s_kn[c] = elem_to_f32<DT>(k);
      }
    }
  if (fresh_key && tid < vdim) {
    const size_t at = (size_t)e * vd + (size_t)g * vdim + tid;
    float v = prow[(size_t)ap.heads * dim + kd + (size_t)g * vdim + tid];
    if (ap.vmode == 1 && appends) ap.vfirst[at] = v;
    if (ap.vmode == 2) { const float lam = ap.lam[0]; v = fmaf(lam, ap.vfirst[at], __fmul_rn(1.0f - lam, v)); }
    const elem_t<DT> sv = f32_to_elem<DT>(v);
    if (appends) {
      const size_t pg = (size_t)tbl[pos >> m.page_shift];
      reinterpret_cast<elem_t<DT>*>(ap.poolV)[((pg << m.page_shift) + (size_t)(pos & pmask)) * vd + (size_t)g * vdim + tid] = sv;
      if (ap.poolVT) reinterpret_cast<elem_t<DT>*>(ap.poolVT)[((pg * vd + (size_t)g * vdim + tid) << m.page_shift) + (size_t)(pos & pmask)] = sv;
    }
    s_vn[tid] = elem_to_f32<DT>(sv);
  }
  __syncthreads();
  // scores
#pragma unroll
  for (int u = 0; u < KW / 4; u++) {
    if (64 * u >= n) break;
    const int i = 4 * (wv + 16 * u) + sub;
    float sc[MG] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 2; c++) {
      if (128 * c >= dim) break;
      const int at = ch + 128 * c;
      float k[8];
      slice_unpack<DT>(kr[u][c], k);
      if (fresh_key && i == n - 1) {
#pragma unroll
        for (int x = 0; x < 8; x++) k[x] = s_kn[min(at + x, dim - 1)];
      }
      if (at < dim) {
#pragma unroll
        for (int r = 0; r < MG; r++) {
          const f32x4 q0 = *reinterpret_cast<const f32x4*>(&s_qr[min(r, nh - 1)][at]), q1 = *reinterpret_cast<const f32x4*>(&s_qr[min(r, nh - 1)][at + 4]);
#pragma unroll
          for (int x = 0; x < 8; x++) sc[r] = fmaf(k[x], x < 4 ? q0[x & 3] : q1[x & 3], sc[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < MG; r++) { sc[r] = row_group_sum<16>(sc[r]); if ((lane & 15) == r && r < nh && i < n) s_s[r][i] = sc[r]; }
  }
  __syncthreads();
  if (wv < nh) {
    const int h = h0 + wv;
    const float slope2 = a.dist_bias ? distance_slope(h, ap.heads) * LOG2E : 0.f;
    float s[STEP_MAX_KEYS / 64], mx = a.has_sink ? a.sink * LOG2E : -INFINITY, l = 0.f;
#pragma unroll
    for (int u = 0; u < STEP_MAX_KEYS / 64; u++) {
      const int i = lane + 64 * u;
      float v = i < n ? s_s[wv][i] : -INFINITY;
      if (capped && i < n) v = a.softcap * tanhf(v / a.softcap) * LOG2E;
      s[u] = i < n ? fmaf(-slope2, (float)(n - 1 - i), v) : -INFINITY;
      mx = fmaxf(mx, s[u]);
    }
    mx = group_max<64>(mx);
    const bool dead = mx == -INFINITY;
#pragma unroll
    for (int u = 0; u < STEP_MAX_KEYS / 64; u++) { const float p = dead ? 0.f : __builtin_amdgcn_exp2f(s[u] - mx); l += p; if (lane + 64 * u < n) s_s[wv][lane + 64 * u] = p; }
    l = wave_sum(l);
    if (a.has_sink) l += __builtin_amdgcn_exp2f(a.sink * LOG2E - mx);
    if (lane == 0) s_l[wv] = l;
  }
  __syncthreads();
  // values
  float acc[MG][2];
#pragma unroll
  for (int r = 0; r < MG; r++) acc[r][0] = acc[r][1] = 0.f;
#pragma unroll
  for (int u = 0; u < KW; u++) {
    if (16 * u >= n) break;
    const int i = wv + 16 * u;
    if (i >= n) break;                                             // (wave-uniform)
    const bool own = fresh_key && i == n - 1;
    const float v0 = own ? s_vn[min(lane, vdim - 1)] : vr[u][0], v1 = own ? s_vn[min(lane + 64, vdim - 1)] : vr[u][1];
#pragma unroll
    for (int r = 0; r < MG; r++) { const float p = s_s[min(r, nh - 1)][i]; acc[r][0] = fmaf(p, v0, acc[r][0]); acc[r][1] = fmaf(p, v1, acc[r][1]); }
  }
#pragma unroll
  for (int r = 0; r < MG; r++)
#pragma unroll
    for (int c = 0; c < 2; c++) if (lane + 64 * c < STEP_MAX_VDIM) s_acc[wv][r][lane + 64 * c] = acc[r][c];
  __syncthreads();
  const int r = tid >> 7, c = tid & 127;                           // (STEP_MAX_VDIM columns a head)
  if (r < nh && c < vdim) {
    const size_t hc = (size_t)(h0 + r) * vdim + c;
    float t[16];
#pragma unroll
    for (int w = 0; w < 16; w++) t[w] = s_acc[w][r][c];
#pragma unroll
    for (int o = 8; o > 0; o >>= 1)
#pragma unroll
      for (int w = 0; w < o; w++) t[w] += t[w + o];
    float v = s_l[r] > 0.f ? t[0] / s_l[r] : 0.f;
    if (a.gate) v = v / (1.0f + expf(-a.gate[(size_t)e * a.ldg + (a.gate_per_head ? (size_t)(h0 + r) : hc)]));
    a.out[(size_t)e * a.ldo + hc] = v * a.out_scale;
  }
}
template <int DT>
__global__ __launch_bounds__(1024) void gqa_group_step_kernel(StepMeta m, GqaStepArgs a) { gqa_group_step_body<DT>(m, a, blockIdx.x, blockIdx.y); }

// both halves of a parallel mixer (attention beside a delta rule) in one launch: grid (entries, heads of the one + heads of the other)
template <int DT, int DPER>
__global__ __launch_bounds__(STEP_THREADS) void parallel_step_kernel(StepMeta m, GqaStepArgs a, RecStepArgs r, const int log_cp) {
  if ((int)blockIdx.y < a.ap.heads) gqa_step_body<DT, STEP_THREADS>(m, a, blockIdx.x, blockIdx.y);
  else rec_step_body<DT_F32, REC_DELTA, DPER>(m, r, log_cp, blockIdx.x, blockIdx.y - a.ap.heads);
}

}  // namespace tgx
