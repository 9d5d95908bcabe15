// Gated DeltaNet step, split path for 5-8 rows: gdn_split_kernel (each value head's 128 state
// columns over 4 workgroups) followed by gdn_finish_kernel (one workgroup per head). Same
// per-column arithmetic as gdn_step_kernel (gdn.hip), so the same bits.
//
// us per call at Hk 16 / Hv 48, n : pending 5:5 12.89 -> 11.97, 6:3 13.39 -> 12.26, 7:0 13.57 -> 11.48,
// 8:8 15.57 -> 14.43 since the per-row work ahead of the recurrence is spread over the waves, same bits
// (before, 4 waves of 8 ran every row's conv, square root and divisions in turn).
//
// This file is compiled with LLVM's max-ILP machine scheduler; the one-workgroup kernel in
// gdn.hip keeps the default. Same-box A/B of the whole Gated DeltaNet source under max-ILP, us
// per call at Hk 16 / Hv 48, before that: 6 rows 15.36 -> 14.63, 8 rows 17.39 -> 16.48 (this path);
// the one-workgroup kernel 1% slower. Same bits.
#include "gdn_common.hpp"

namespace qe {

// ------------------------------------------------------------------ split kernels
// The same step with each head's 128 state columns split over GDN_SPLIT workgroups of 512
// threads (32 columns each): four times the CUs for the state I/O and the delta-rule VALU work,
// which bound the one-workgroup kernel. Each workgroup holds rows 8 rg .. +7 of its columns per
// lane and runs the same per-column arithmetic, so the state is bit-identical to the
// one-workgroup kernel's. Every workgroup repeats the conv, l2norm and gates of its head's q and
// k (256 channels) and does the v channels of its own columns.
//
// Nothing waits across workgroups. What needs a whole head (the gated RMSNorm sums the squares
// of a row's 128 outputs) or must not overwrite what another part still reads (the staged k rows
// and gates of the previous call, which every part of a head replays) is left to a second
// kernel, gdn_finish_kernel: gdn_split_kernel writes each row's outputs o, already bf16 values,
// into `out` unnormalised, and stages only its own v columns; gdn_finish_kernel (one workgroup
// per head, after every part has finished) recomputes the head's normalised k rows and gates with
// the same arithmetic, stages them, and normalises `out` in place. Block b runs head b % Hv, part
// b / Hv: with Hv a multiple of 8 the parts of a head share an XCD.

// Eight waves, two per SIMD (one wave's reduction and LDS latencies hide behind the other's), one
// state column per lane. Before the recurrence a call is a chain of latencies, so its per-row work
// is spread over the waves: the conv rows 0-3 of the 256 q and k channels run on waves 0-3 and rows
// 4-7 on waves 4-7, the v channels one (row, channel) per lane of waves 4-7, and a row's
// 1 / sqrt(sum of squares) is computed by one lane and broadcast. The recurrence reads the next
// step's rows from LDS ahead of the current step's arithmetic.

// One step's operands of a lane: rows 8 rg .. +7 of k (and q), its column of v, and the gates.
struct DeltaRow {
  float k[8], q[8], v[1], decay, beta;
};
__device__ __forceinline__ void delta_row_k(DeltaRow& d, const float* k_row, const float* v_row,
                                            const float* g_row, int rg, int lc) {
  lds_read8(k_row + rg * 8, d.k);
  d.v[0] = v_row[lc];
  d.decay = g_row[0];
  d.beta = g_row[1];
}

__global__ void __launch_bounds__(GDN_SPLIT_THREADS)
gdn_split_kernel(const __bf16* __restrict__ qkv, const __bf16* __restrict__ b,
                 const __bf16* __restrict__ a, long ldp, __bf16* __restrict__ ring,
                 const __bf16* __restrict__ conv_w, const __bf16* __restrict__ A_log,
                 const __bf16* __restrict__ dt_bias, float* __restrict__ S,
                 float* __restrict__ st_k, float* __restrict__ st_v, float* __restrict__ st_g,
                 const int* __restrict__ ctl, __bf16* __restrict__ out, long ldo, int n, int Hk,
                 int Hv) {
  constexpr int CW = GDN_SPLIT_COLS;
  constexpr int RH = GDN_MAXN / 2;  // conv rows per thread
  static_assert(GDN_SPLIT_THREADS == 2 * 2 * GDN_D && CW == 32, "two halves of 256 q/k channels");
  __shared__ __align__(16) float srow[GDN_MAXN * (GDN_D + CW)];  // replayed rows
  float (*sk)[GDN_D] = reinterpret_cast<float (*)[GDN_D]>(srow);
  float (*sv)[CW] = reinterpret_cast<float (*)[CW]>(srow + GDN_MAXN * GDN_D);
  __shared__ __align__(16) float qa[GDN_MAXN][GDN_D], ka[GDN_MAXN][GDN_D], va[GDN_MAXN][CW];
  __shared__ __align__(16) float oa[GDN_MAXN][CW];
  __shared__ float sg[GDN_MAXN][2], ga[GDN_MAXN][2], l2p[GDN_MAXN][4];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = blockIdx.x % Hv, g = blockIdx.x / Hv;
  const int r = Hv / Hk, i = j / r;
  const int C = 2 * Hk * GDN_D + Hv * GDN_D;
  const int cb = g * CW;                              // first state column of this workgroup
  const int rg = lane >> 2, lc = 4 * w + (lane & 3);  // rows 8 rg .. +7 of column lc
  float* Sj = S + (size_t)j * GDN_D * GDN_D;

  // Loads, all unconditional with in-bounds indices (as in the one-workgroup kernel).
  const int P = ctl[0];
  const int pend = min(max(ctl[1], 0), GDN_MAXN);
  const int t0 = RH * (w >> 2);                       // this thread's conv rows t0 .. t0 + 3
  const int part = (w >> 1) & 1, c = tid & 127;       // q (part 0) or k (part 1) channel c
  const int ch = (part * Hk + i) * GDN_D + c;
  const int tv = (tid >> 5) & 7, cv = tid & (CW - 1);  // (row, v channel) of threads 256 ..
  const int chv = 2 * Hk * GDN_D + j * GDN_D + cb + cv;
  const uint2 wq = *reinterpret_cast<const uint2*>(conv_w + (size_t)ch * 4);
  const uint2 wvv = *reinterpret_cast<const uint2*>(conv_w + (size_t)chv * 4);
  __bf16 xb[3 + RH], xbv[4];
#pragma unroll
  for (int q = 3; q < 3 + RH; ++q) xb[q] = conv_input(qkv, ldp, ring, C, P, n, t0 + q - 3, ch);
  const int gt = tid - (GDN_SPLIT_THREADS - WAVE);    // gate row of the last wave's first n threads
  const int gtc = min(max(gt, 0), n - 1);
  const __bf16 bb = b[(size_t)gtc * ldp + j], ab = a[(size_t)gtc * ldp + j];
  const __bf16 dtb = dt_bias[j], alb = A_log[j];
  const bool first = tid < 2 * GDN_D;                 // threads that move 256-thread pieces
  const int ot = (tid >> 5) & 7, oc = tid & (CW - 1);  // output element (row ot, column cb + oc)
#pragma unroll
  for (int q = 0; q < 3; ++q) xb[q] = conv_input(qkv, ldp, ring, C, P, n, t0 + q - 3, ch);
#pragma unroll
  for (int q = 0; q < 4; ++q) xbv[q] = conv_input(qkv, ldp, ring, C, P, n, tv + q - 3, chv);
  // Staged rows, a 16-byte piece per thread: k (waves 0-3) or v columns of this part (the last
  // waves move the same 64 pieces). No branch: the compiler sinks a load that only a branch uses
  // into it, behind the state's loads, and the wait for it there is a wait for the state.
  const int vr = (tid >> 3) & 7, vp = tid & 7;  // staged v: row vr, columns cb + 4 vp ..
  const F4 stp = *reinterpret_cast<const F4*>(
      w < 4 ? st_k + ((size_t)ot * Hv + j) * GDN_D + 4 * oc
            : st_v + ((size_t)vr * Hv + j) * GDN_D + cb + 4 * vp);
  const float2 stg = *reinterpret_cast<const float2*>(st_g + ((size_t)(tid & 7) * Hv + j) * 2);
  float s[8][1];
#pragma unroll
  for (int rr = 0; rr < 8; ++rr) s[rr][0] = Sj[(size_t)(rg * 8 + rr) * GDN_D + cb + lc];

  *reinterpret_cast<F4*>(w < 4 ? &sk[ot][4 * oc] : &sv[vr][4 * vp]) = stp;
  if (tid < GDN_MAXN) {
    sg[tid][0] = stg.x;
    sg[tid][1] = stg.y;
  }
  float y[RH];
  {
    const bool head_writer = g == 0 && j % r == 0;  // one writer of the shared q/k ring slots
    const float cw[4] = {lo_bf16(wq.x), hi_bf16(wq.x), lo_bf16(wq.y), hi_bf16(wq.y)};
    float xs[3 + RH];
#pragma unroll
    for (int q = 0; q < 3 + RH; ++q) xs[q] = conv_value(xb[q], P, t0 + q - 3);
#pragma unroll
    for (int t = 0; t < RH; ++t) {
      y[t] = 0.f;
      if (t0 + t < n) {
        y[t] = conv_silu(cw, xs, t);
        if (head_writer) ring[(size_t)((P + t0 + t) & (GDN_RING - 1)) * C + ch] = xb[3 + t];
        const float ss = wave_sum_fast(y[t] * y[t]);  // q: waves 0, 1 mod 4; k: waves 2, 3 mod 4
        if (lane == 0) l2p[t0 + t][w & 3] = ss;
      }
    }
  }
  if (!first && tv < n) {  // the v channels of this workgroup's columns
    const float cw[4] = {lo_bf16(wvv.x), hi_bf16(wvv.x), lo_bf16(wvv.y), hi_bf16(wvv.y)};
    float xs[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) xs[q] = conv_value(xbv[q], P, tv + q - 3);
    va[tv][cv] = conv_silu(cw, xs, 0);
    ring[(size_t)((P + tv) & (GDN_RING - 1)) * C + chv] = xbv[3];
  }
  if (gt >= 0 && gt < n) {
    const float2 gv = gate_values(bb, ab, dtb, alb);
    ga[gt][0] = gv.x;
    ga[gt][1] = gv.y;
  }
  __syncthreads();

  // Stage this call's v columns for the next call (after the barrier: this workgroup's reads of
  // the previous call's rows at the same addresses are in LDS by now; no other workgroup reads
  // these columns). The k rows and gates, which every part of the head reads, are staged by
  // gdn_finish_kernel.
  if (first && ot < n) st_v[((size_t)ot * Hv + j) * GDN_D + cb + oc] = va[ot][oc];
  if (t0 < n) {
    const float sqrt_dk = 11.313708498984761f;  // sqrt(128) rounded to fp32
    const int tl = min(t0 + (lane & (RH - 1)), n - 1);
    const float inv_l = 1.0f / sqrtf((l2p[tl][2 * part] + l2p[tl][2 * part + 1]) + 1e-6f);
#pragma unroll
    for (int t = 0; t < RH; ++t) {
      const float inv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv_l), t));
      if (part == 0)
        qa[t0 + t][c] = (y[t] * inv) / sqrt_dk;
      else
        ka[t0 + t][c] = y[t] * inv;
    }
  }

  // ---- 1. replay, write the committed columns back ----
  if (pend > 0) {
    DeltaRow d[2];
    delta_row_k(d[0], sk[0], sv[0], sg[0], rg, lc);
#pragma unroll 2
    for (int t = 0; t < pend; ++t) {
      const int tn = min(t + 1, GDN_MAXN - 1);
      delta_row_k(d[1], sk[tn], sv[tn], sg[tn], rg, lc);
      delta_step(s, d[0].k, d[0].v, d[0].decay, d[0].beta);
      d[0] = d[1];
    }
#pragma unroll
    for (int rr = 0; rr < 8; ++rr) Sj[(size_t)(rg * 8 + rr) * GDN_D + cb + lc] = s[rr][0];
  }
  lds_barrier();  // q and k whole (the state's stores need not have arrived)

  // ---- 2. new rows on the register copy ----
  DeltaRow d[2];
  delta_row_k(d[0], ka[0], va[0], ga[0], rg, lc);
  lds_read8(&qa[0][rg * 8], d[0].q);
#pragma unroll 2
  for (int t = 0; t < n; ++t) {
    const int tn = min(t + 1, n - 1);
    delta_row_k(d[1], ka[tn], va[tn], ga[tn], rg, lc);
    lds_read8(&qa[tn][rg * 8], d[1].q);
    float o[1];
    delta_step(s, d[0].k, d[0].v, d[0].decay, d[0].beta);
    read_out(s, d[0].q, o);
    if (rg == 0) oa[t][lc] = o[0];
    d[0] = d[1];
  }
  lds_barrier();

  // ---- 3. this workgroup's columns of each row's output, unnormalised (o is a bf16 value, so
  // `out` holds it exactly); gdn_finish_kernel normalises the whole row ----
  if (first && ot < n) out[(size_t)ot * ldo + j * GDN_D + cb + oc] = f32_to_bf16(oa[ot][oc]);
}

// Second kernel of a split call, one 512-thread workgroup per value head j, after every part of
// gdn_split_kernel has finished (so no part still reads the previous call's staged rows):
//   * threads 128 p .. 128 p + 127 recompute the normalised k channels of rows 2p and 2p + 1
//     (conv + SiLU from the ring history and the input rows, the sum of squares of the even and
//     the odd wave added in that order, as gdn_split_kernel adds it) and stage them; the last
//     wave's first n threads stage the gates;
//   * wave w normalises row w of the head's outputs in place (gated_norm_row).
__global__ void __launch_bounds__(GDN_FINISH_THREADS)
gdn_finish_kernel(const __bf16* __restrict__ qkv, const __bf16* __restrict__ z,
                  const __bf16* __restrict__ b, const __bf16* __restrict__ a, long ldp,
                  const __bf16* __restrict__ ring, const __bf16* __restrict__ conv_w,
                  const __bf16* __restrict__ A_log, const __bf16* __restrict__ dt_bias,
                  const __bf16* __restrict__ norm_w, float* __restrict__ st_k,
                  float* __restrict__ st_g, const int* __restrict__ ctl, __bf16* __restrict__ out,
                  long ldo, int n, int Hk, int Hv, float eps) {
  constexpr int RQ = GDN_MAXN * GDN_D / GDN_FINISH_THREADS;  // k rows per thread
  static_assert(GDN_FINISH_THREADS == GDN_MAXN * WAVE && RQ == 2, "a wave per row");
  __shared__ __align__(16) float oa[GDN_MAXN][GDN_D];
  __shared__ float l2p[GDN_MAXN][2];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = blockIdx.x, i = j / (Hv / Hk);
  const int C = 2 * Hk * GDN_D + Hv * GDN_D;
  const int P = ctl[0];
  const int c = tid & 127, t0 = RQ * (w >> 1);
  const int ch = (Hk + i) * GDN_D + c;  // k channel c of qk head i
  const uint2 wk = *reinterpret_cast<const uint2*>(conv_w + (size_t)ch * 4);
  // outputs, z and weights of row w, columns 2 lane, 2 lane + 1
  const int tw = min(w, n - 1);
  const __bf16* op = out + (size_t)tw * ldo + j * GDN_D + 2 * lane;
  const __bf16* zp = z + (size_t)tw * ldp + j * GDN_D + 2 * lane;
  const __bf16 ob0 = op[0], ob1 = op[1], zb0 = zp[0], zb1 = zp[1];
  const float nw0 = bf16_to_f32(norm_w[2 * lane]), nw1 = bf16_to_f32(norm_w[2 * lane + 1]);
  const int gt = tid - (GDN_FINISH_THREADS - WAVE);
  const int gtc = min(max(gt, 0), n - 1);
  const __bf16 bb = b[(size_t)gtc * ldp + j], ab = a[(size_t)gtc * ldp + j];
  const __bf16 dtb = dt_bias[j], alb = A_log[j];
  __bf16 xb[3 + RQ];
#pragma unroll
  for (int q = 0; q < 3 + RQ; ++q) xb[q] = conv_input(qkv, ldp, ring, C, P, n, t0 + q - 3, ch);

  oa[w][2 * lane] = bf16_to_f32(ob0);
  oa[w][2 * lane + 1] = bf16_to_f32(ob1);
  const float cw[4] = {lo_bf16(wk.x), hi_bf16(wk.x), lo_bf16(wk.y), hi_bf16(wk.y)};
  float xs[3 + RQ], y[RQ];
#pragma unroll
  for (int q = 0; q < 3 + RQ; ++q) xs[q] = conv_value(xb[q], P, t0 + q - 3);
#pragma unroll
  for (int t = 0; t < RQ; ++t) {  // both rows also at t0 + t = n: no load behind a branch
    y[t] = conv_silu(cw, xs, t);
    const float ss = wave_sum_fast(y[t] * y[t]);
    if (lane == 0) l2p[t0 + t][w & 1] = ss;
  }
  const float sz0 = silu_f(bf16_to_f32(zb0)), sz1 = silu_f(bf16_to_f32(zb1));
  __syncthreads();
#pragma unroll
  for (int t = 0; t < RQ; ++t) {
    if (t0 + t < n) {
      const float inv = 1.0f / sqrtf((l2p[t0 + t][0] + l2p[t0 + t][1]) + 1e-6f);
      st_k[((size_t)(t0 + t) * Hv + j) * GDN_D + c] = y[t] * inv;
    }
  }
  if (gt >= 0 && gt < n)
    *reinterpret_cast<float2*>(st_g + ((size_t)gt * Hv + j) * 2) = gate_values(bb, ab, dtb, alb);
  if (w < n)
    gated_norm_row(oa[w], lane, nw0, nw1, sz0, sz1, eps,
                   out + (size_t)w * ldo + j * GDN_D);
}

hipError_t launch_gdn_split(const __bf16* qkv, const __bf16* z, const __bf16* b, const __bf16* a,
                            long ldp, __bf16* ring, const __bf16* conv_w, const __bf16* A_log,
                            const __bf16* dt_bias, const __bf16* norm_w, float* S, float* st_k,
                            float* st_v, float* st_g, const int* ctl, __bf16* out, long ldo,
                            int n, int Hk, int Hv, float eps, hipStream_t stream) {
  gdn_split_kernel<<<dim3(Hv * GDN_SPLIT), dim3(GDN_SPLIT_THREADS), 0, stream>>>(
      qkv, b, a, ldp, ring, conv_w, A_log, dt_bias, S, st_k, st_v, st_g, ctl, out, ldo, n, Hk, Hv);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  gdn_finish_kernel<<<dim3(Hv), dim3(GDN_FINISH_THREADS), 0, stream>>>(qkv, z, b, a, ldp, ring, conv_w, A_log,
                                                        dt_bias, norm_w, st_k, st_g, ctl, out,
                                                        ldo, n, Hk, Hv, eps);
  return hipGetLastError();
}

}  // namespace qe
