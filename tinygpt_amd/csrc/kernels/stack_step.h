// stack_step.h — one decoded token of a mixer in ONE launch: what stands between the mixer's products.  First the recurrences, then attention over a short context.  A step of single tokens is bound by its launches (2.6 us for an
// empty one), and a recurrence took three to five of them: the low-rank decay's second product or the convolution with its norms and gates, the rotation, the scan, the norm and gate
// behind it.  Here a workgroup owns a head of one entry with all of its value columns, so that nothing crosses workgroups: the head's inputs are made in LDS, the state [dim][vdim]
// passes through the registers of 1024 threads once (rows of it are read and written whole, 256 bytes a wave and row; the scan's workgroups of sixteen columns take 64-byte
// pieces) and is on its way before anything else is computed, and the outputs are normed and gated where they are.
// The arithmetic is that of the kernels it stands for (stack_rec.h, stack_seq.h), fp32 throughout; sums over the key channels and over a head's outputs meet in another order.
//
// Threads: column j = tid & (CP - 1) (CP: vdim rounded up to a power of two), row group tid / CP with DPER rows each.
// Measured, us a launch in a decoded step's trace (before: the launches that it stands for): one stream, delta rule of 8 heads of 128 x 128 7.4 (convolution 3.9, scan 5.3, norm 2.6),
// wkv of 16 heads of 64 x 64 with its decays 5.2 (3.8, 4.1, 2.5); sixteen entries, channel decays of 8 heads of 128 x 128 9.7 (5.4, 11.7, 3.3), retention of 4 heads of 128 x 256 with
// its rotation 9.3 (3.7, 9.3, 3.0; with the inputs held in registers, which spill at 32 rows a lane, 17.5).
#pragma once
#include "stack_rec.h"
#include "stack_seq.h"

namespace tgx {

constexpr int STEP_MAX_DIM = 256, STEP_MAX_TAPS = 8;
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
  __shared__ __attribute__((aligned(16))) float s_q[STEP_MAX_DIM + 8], s_k[STEP_MAX_DIM + 8], s_w[STEP_MAX_DIM + 8];      // (zeros behind dim)
  __shared__ float s_v[STEP_MAX_DIM], s_b[2], s_n[16], s_unit[2];
  __shared__ float s_pk[1024], s_po[1024];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int t = e, row = m.tok_row[t], pos = m.tok_pos[t], par = m.tok_par[t];      // (an entry is a token)
  const int dim = a.s.dim, vdim = a.s.vdim, share = a.s.heads / a.s.kv_heads, kh = h / share;
  const int cp = 1 << log_cp, RG = 1024 >> log_cp, j = tid & (cp - 1), rg = tid >> log_cp, d0 = rg * DPER;
  const bool col = j < vdim;
  float* Sg = a.s.S + ((size_t)row * a.s.heads + h) * (size_t)dim * vdim;
  float S[DPER], ub[KIND == REC_WKV ? DPER : 1];
#pragma unroll
  for (int dd = 0; dd < DPER; dd++) {
    const int d = d0 + dd;
    S[dd] = (pos != 0 && d < dim && col) ? Sg[(size_t)d * vdim + j] : 0.f;
    if (KIND == REC_WKV) ub[dd] = d < dim ? a.s.u[(size_t)h * dim + d] : 0.f;
  }
  // ---- the head's inputs
  if (tid < 8) s_q[dim + tid] = s_k[dim + tid] = s_w[dim + tid] = 0.f;
  if (KIND != REC_WKV && a.prep) {
    const DeltaPrepArgs& p = a.p;
    const int GD = p.kv_heads * dim, C = 2 * GD + p.heads * vdim, nb = p.taps - 1;
    if (tid < 2 * dim + vdim) {
      const int part = tid < dim ? 0 : tid < 2 * dim ? 1 : 2, cc = tid - part * dim, c = part == 0 ? kh * dim + cc : part == 1 ? GD + kh * dim + cc : 2 * GD + h * vdim + cc;
      const float* st_old = p.state + (size_t)par * p.state_buf + (size_t)row * nb * C + c;
      float* st_new = p.state + (size_t)(par ^ 1) * p.state_buf + (size_t)row * nb * C + c;
      const float* cw = p.cw + (size_t)c * p.taps;
      const float x0 = p.proj[(size_t)t * p.ldp + p.col0 + c];
      float old[STEP_MAX_TAPS - 1];                                // old[d - 1]: the row d positions back
#pragma unroll
      for (int d = 1; d < STEP_MAX_TAPS; d++) old[d - 1] = d <= nb && pos - d >= 0 ? st_old[(size_t)(nb - d) * C] : 0.f;
      float acc = cw[nb] * x0;
#pragma unroll
      for (int d = 1; d < STEP_MAX_TAPS; d++) if (d <= nb) acc = fmaf(cw[nb - d], old[d - 1], acc);
      const float act = acc / (1.0f + expf(-acc));
      if (part == 0) s_q[cc] = act; else if (part == 1) s_k[cc] = act; else s_v[cc] = act;
      if (nb > 0 && (part == 2 || h == kh * share)) {              // (heads that share keys: the first of them moves the tails)
        st_new[(size_t)(nb - 1) * C] = x0;
#pragma unroll
        for (int d = 1; d < STEP_MAX_TAPS - 1; d++) if (d < nb) st_new[(size_t)(nb - 1 - d) * C] = old[d - 1];
      }
    }
    if (tid == 1023) {
      const float* pr = p.proj + (size_t)t * p.ldp + p.col0;
      s_b[0] = 1.0f / (1.0f + expf(-pr[p.b_col + h]));
      if (p.a_log) {
        const float za = pr[p.b_col + p.heads + h] + p.dt_bias[h];
        const float sp = za > 20.f ? za : log1pf(expf(za));
        s_b[1] = expf(-expf(p.a_log[h]) * sp);
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
    } else if (tid >= 512 && tid < 512 + vdim) s_v[tid - 512] = a.s.v[(size_t)t * a.s.ldv + (size_t)h * vdim + tid - 512];
    if (KIND != REC_WKV && tid == 1023) {
      const size_t at = (size_t)t * a.s.ldg + h;
      if (KIND == REC_SSD && a.s.fixed) { s_b[0] = a.s.beta0; s_b[1] = a.s.fixed[h]; }
      else { s_b[0] = a.s.beta[at]; if (KIND != REC_CDELTA) s_b[1] = a.s.g[at]; }
    }
    if (KIND == REC_WKV && a.w2) {                                 // sixteen lanes a channel
      const elem_t<DT>* w2 = reinterpret_cast<const elem_t<DT>*>(a.w2);
      for (int c0 = 0; c0 < dim; c0 += 64) {
        const int c = c0 + (tid >> 4);
        float acc = 0.f;
        for (int r = tid & 15; r < a.rank; r += 16)
          acc = fmaf(elem_to_f32<DT>(w2[((size_t)h * dim + min(c, dim - 1)) * a.rank + r]), round_storage_if<DT>(a.lora[(size_t)t * a.ldlora + r], a.terms == 1), acc);
        acc = row_group_sum<16>(acc);
        if ((tid & 15) == 0 && c < dim) s_w[c] = expf(-expf(acc + a.w0[(size_t)h * dim + c]));
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
  const bool mine = tid < vdim;
  const float gate = mine ? a.g.gate[(size_t)t * a.g.ldg + (size_t)h * vdim + tid] : 0.f, w = mine && a.g.w ? a.g.w[(size_t)h * a.g.w_hstride + tid] : 1.f;
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
  a.g.out[(size_t)t * a.g.ldo + (size_t)h * vdim + tid] = o * rinv * w * (a.g.silu_gate ? gate * sg : sg);
}

template <int DT, int KIND, int DPER>
__global__ __launch_bounds__(1024) void rec_step_kernel(StepMeta m, RecStepArgs a, const int log_cp) { rec_step_body<DT, KIND, DPER>(m, a, log_cp, blockIdx.x, blockIdx.y); }

// ---- attention of single tokens over up to STEP_MAX_KEYS keys, the token's own among them.  The divided form took three launches for this (append, a walk of key tiles by matrix
// instructions, merge), the undivided one two, its walk a chain of 1.3 us a tile on a workgroup per key / value head.  Here a workgroup of sixteen waves owns an entry and a key /
// value head with its (up to four) query heads: it finishes the token's queries, key and value in LDS (gqa_append_kernel) and stores the latter two, then
//   scores   four keys a wave at a time, sixteen lanes a key with eight channels each; every wave's keys are on their way at once
//   softmax  a wave per query head, base 2, as in gqa_attn_mfma_kernel (cap, distance slope, sink, mask)
//   values   a key per wave at a time, a lane's channels of all query heads; the waves' sums meet in LDS
// Queries and probabilities stay fp32 (the matrix forms take them as two 16-bit terms).
// Measured, us: one stream of 50 to 95 keys, two key / value heads of 128 x 128 7.9 (append 3.0, undivided walk 7.9; 8.4 with the columns of a row found by divisions); beside a delta rule in one launch 9.0 (7.4 of the rule's own).
constexpr int STEP_MAX_KEYS = 256, STEP_MAX_GROUP = 4, STEP_MAX_VDIM = 128;
struct GqaStepArgs {
  GqaAppendArgs ap;          // the token's row (maps 1, no q_hi, no qk_unit_eps)
  const float* gate; long long ldg; int gate_per_head;
  float* out; long long ldo; float out_scale;
  float scale, sink; int has_sink;
  int mask_kind, mask_size;
  float softcap; int dist_bias;
  const void *poolK, *poolV; // the pools that are read (those of ap where the layer appends)
};
template <int DT>
__device__ __forceinline__ void gqa_step_body(const StepMeta& m, const GqaStepArgs& a, const int e, const int g) {
  constexpr int MG = STEP_MAX_GROUP, KW = STEP_MAX_KEYS / 16;      // keys of a wave
  constexpr float LOG2E = 1.4426950408889634f;
  __shared__ __attribute__((aligned(16))) float s_qr[MG][STEP_MAX_DIM], s_kn[STEP_MAX_DIM];
  __shared__ float s_vn[STEP_MAX_VDIM], s_s[MG][STEP_MAX_KEYS], s_l[MG], s_acc[16][MG][STEP_MAX_VDIM];
  const GqaAppendArgs& ap = a.ap;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = m.tok_row[e], pos = m.tok_pos[e], dim = ap.dim, vdim = ap.vdim, Gq = ap.heads / ap.kv_heads;
  const int lo = first_key(pos, a.mask_kind, a.mask_size), n = pos - lo + 1, kd = ap.kv_heads * dim, vd = ap.kv_heads * vdim;
  const int* tbl = m.tbl + (size_t)row * m.tbl_stride;
  const bool fresh_key = ap.poolK != nullptr;                      // (a layer that reads another layer's pool appends nothing: its last key stands there)
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
  const int nq = Gq + (fresh_key ? 1 : 0);
  if (wv < 2 * nq)                                                 // two waves a row
    for (int c = lane + 64 * (wv & 1); c < dim; c += 128) {
      const int r = wv >> 1;
      const float* u = prow + (r < Gq ? (size_t)(g * Gq + r) * dim : (size_t)ap.heads * dim + (size_t)g * dim);
      float v = u[c];
      if (c < ap.rot_dims) {
        const int half = ap.rot_dims >> 1, p = ap.rot_pairs ? c >> 1 : c < half ? c : c - half;
        const bool first = ap.rot_pairs ? (c & 1) == 0 : c < half;
        const float cs = ap.cs[((size_t)pos * half + p) * 2], sn = ap.cs[((size_t)pos * half + p) * 2 + 1], o = u[ap.rot_pairs ? c ^ 1 : first ? c + half : c - half];
        v = first ? __fsub_rn(__fmul_rn(v, cs), __fmul_rn(o, sn)) : __fadd_rn(__fmul_rn(v, cs), __fmul_rn(o, sn));
      }
      if (r < Gq) s_qr[r][c] = v * temp * qscale;
      else {
        const elem_t<DT> k = f32_to_elem<DT>(v);
        reinterpret_cast<elem_t<DT>*>(ap.poolK)[(((size_t)tbl[pos >> m.page_shift] << m.page_shift) + (size_t)(pos & pmask)) * kd + (size_t)g * dim + c] = k;
        s_kn[c] = elem_to_f32<DT>(k);
      }
    }
  if (fresh_key && tid < vdim) {
    const size_t at = (size_t)e * vd + (size_t)g * vdim + tid;
    float v = prow[(size_t)ap.heads * dim + kd + (size_t)g * vdim + tid];
    if (ap.vmode == 1) ap.vfirst[at] = v;
    if (ap.vmode == 2) { const float lam = ap.lam[0]; v = fmaf(lam, ap.vfirst[at], __fmul_rn(1.0f - lam, v)); }
    const elem_t<DT> sv = f32_to_elem<DT>(v);
    const size_t pg = (size_t)tbl[pos >> m.page_shift];
    reinterpret_cast<elem_t<DT>*>(ap.poolV)[((pg << m.page_shift) + (size_t)(pos & pmask)) * vd + (size_t)g * vdim + tid] = sv;
    if (ap.poolVT) reinterpret_cast<elem_t<DT>*>(ap.poolVT)[((pg * vd + (size_t)g * vdim + tid) << m.page_shift) + (size_t)(pos & pmask)] = sv;
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
          const f32x4 q0 = *reinterpret_cast<const f32x4*>(&s_qr[min(r, Gq - 1)][at]), q1 = *reinterpret_cast<const f32x4*>(&s_qr[min(r, Gq - 1)][at + 4]);
#pragma unroll
          for (int x = 0; x < 8; x++) sc[r] = fmaf(k[x], x < 4 ? q0[x & 3] : q1[x & 3], sc[r]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < MG; r++) { sc[r] = row_group_sum<16>(sc[r]); if ((lane & 15) == r && r < Gq && i < n) s_s[r][i] = sc[r]; }
  }
  __syncthreads();
  if (wv < Gq) {
    const int h = g * Gq + wv;
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
    for (int r = 0; r < MG; r++) { const float p = s_s[min(r, Gq - 1)][i]; acc[r][0] = fmaf(p, v0, acc[r][0]); acc[r][1] = fmaf(p, v1, acc[r][1]); }
  }
#pragma unroll
  for (int r = 0; r < MG; r++)
#pragma unroll
    for (int c = 0; c < 2; c++) if (lane + 64 * c < STEP_MAX_VDIM) s_acc[wv][r][lane + 64 * c] = acc[r][c];
  __syncthreads();
  const int r = tid >> 7, c = tid & 127;                           // (STEP_MAX_VDIM columns a head)
  if (r < Gq && c < vdim) {
    const size_t hc = (size_t)(g * Gq + r) * vdim + c;
    float t[16];
#pragma unroll
    for (int w = 0; w < 16; w++) t[w] = s_acc[w][r][c];
#pragma unroll
    for (int o = 8; o > 0; o >>= 1)
#pragma unroll
      for (int w = 0; w < o; w++) t[w] += t[w + o];
    float v = s_l[r] > 0.f ? t[0] / s_l[r] : 0.f;
    if (a.gate) v = v / (1.0f + expf(-a.gate[(size_t)e * a.ldg + (a.gate_per_head ? (size_t)(g * Gq + r) : hc)]));
    a.out[(size_t)e * a.ldo + hc] = v * a.out_scale;
  }
}
template <int DT>
__global__ __launch_bounds__(1024) void gqa_step_kernel(StepMeta m, GqaStepArgs a) { gqa_step_body<DT>(m, a, blockIdx.x, blockIdx.y); }

// both halves of a parallel mixer (attention beside a delta rule) in one launch: grid (entries, key / value heads of the one + heads of the other)
template <int DT, int DPER>
__global__ __launch_bounds__(1024) void parallel_step_kernel(StepMeta m, GqaStepArgs a, RecStepArgs r, const int log_cp) {
  if ((int)blockIdx.y < a.ap.kv_heads) gqa_step_body<DT>(m, a, blockIdx.x, blockIdx.y);
  else rec_step_body<DT_F32, REC_DELTA, DPER>(m, r, log_cp, blockIdx.x, blockIdx.y - a.ap.kv_heads);
}

}  // namespace tgx
