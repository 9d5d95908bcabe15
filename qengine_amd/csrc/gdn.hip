// Gated DeltaNet decode / verify step on gfx950: n = 1..8 new rows per layer call with lazy
// rollback (reference csrc/gdn.cu:1-25,65-311; math of python/qengine/reference.py:211-242).
//
// Per value head j (qk head i = j / (Hv/Hk)), with the committed fp32 state S_j [128][128] being
// the state after position pos - pending:
//   1. replay: the `pending` rows staged by the previous call (normalised k, v, decay, beta) are
//      applied to S_j, which is written back once;
//   2. new rows t < n at positions pos + t: causal conv (4 taps) + SiLU over the 384 channels of
//      this head, gates, l2norm of q and k, the delta-rule update on a register copy of S_j, and
//      the gated RMSNorm output; their (k, v, decay, beta) are staged for the next call, S_j is
//      not advanced by them.
// The same inline update runs for replayed and new rows, so the committed state after any
// pattern of calls with kept prefixes equals plain one-row decoding bit for bit.
//
// Two paths share the per-column arithmetic (gdn_common.hpp) and so give the same bits:
// gdn_step_kernel (one workgroup per head, below) for 1-4 rows, and gdn_split_kernel (each head
// over 4 workgroups) followed by gdn_finish_kernel (gdn_split.hip) for 5-8 rows.
//
// gfx950 layout: one workgroup of 1024 threads (16 waves, four per SIMD) per value head. Wave w
// owns state columns 8w .. 8w + 7 and lane l holds rows 8(l>>2) .. +7 of columns 8w + 2(l&3), +1
// (16 fp32 registers). The dot products over the 128 state rows are a per-lane 8-term FMA chain
// followed by a butterfly over the 16 lanes that share a column pair (DPP xor 8 / 4, permlane16 / 32
// swaps), so the recurrence needs no LDS and no barrier, and kv, delta and o never leave the wave.
// Three barriers per call, for LDS alone (stores to memory are not waited for): after the per-call
// inputs are in LDS, after the replay (by then q and k are normalised in LDS, once per channel), and
// before the gated RMSNorm, which needs the 128 outputs of a row.
//
// What bounds a short call is the chain of latencies ahead of the first barrier, so the waves take
// roles: waves 0-11 load and convolve (position, then the ring's history, then the arithmetic),
// waves 12-15 bring the state and the staged rows to LDS by DMA meanwhile and hold the gates and the
// output norm's operands. With one role for all, the compiler sank the state's loads below the conv
// and the staged rows' loads into their branch, and the two latencies added up. us per call at
// Hk 16 / Hv 48, n : pending 1:0 6.13 -> 5.45, 2:2 8.18 -> 7.80, 4:0 9.68 -> 8.60, 4:4 11.12 -> 10.79,
// same bits. (A lane's rows straight from memory read 32 bytes of each line per wave: 8.41 against
// 7.73 at one row when the copy through LDS came in.) From there on a row costs ~1 us of one CU's
// VALU: the four waves of a SIMD issue ~125 instructions each for it.
//
// Conv history is a ring of 16 slots [16][C] keyed by absolute position (slot = pos & 15). A call
// reads positions < pos from the ring (negative positions read as 0) and earlier rows of this
// call from its own inputs, and writes the slots of positions pos .. pos+n-1. With n <= 8 the
// read slots (pos-3 .. pos-1) and the written ones never alias, so workgroups sharing a qk head
// need no synchronisation; only the workgroup with j % (Hv/Hk) == 0 writes the q/k channels.
#include "gdn_common.hpp"
#include "qe_gdn.h"

namespace qe {

// Waves 0-11 of the 16: the conv of rows w / 6 and w / 6 + 2 (q, k and v take two waves each);
// waves 12-15: loads. RH: rows per conv thread, 1 for 1-2 rows and 2 for 3-4.
constexpr int CONV_WAVES = 12, LOAD_WAVES = GDN_THREADS / WAVE - CONV_WAVES;
static_assert(GDN_SPLIT_MIN_ROWS - 1 <= LOAD_WAVES, "a wave of the norm per row");

template <int RH>
__global__ void __launch_bounds__(GDN_THREADS)
gdn_step_kernel(const __bf16* __restrict__ qkv, const __bf16* __restrict__ z,
                const __bf16* __restrict__ b, const __bf16* __restrict__ a, long ldp,
                __bf16* __restrict__ ring, const __bf16* __restrict__ conv_w,
                const __bf16* __restrict__ A_log, const __bf16* __restrict__ dt_bias,
                const __bf16* __restrict__ norm_w, float* __restrict__ S,
                float* __restrict__ st_k, float* __restrict__ st_v, float* __restrict__ st_g,
                const int* __restrict__ ctl, __bf16* __restrict__ out, long ldo, int n, int Hk,
                int Hv, float eps) {
  constexpr int MAXN = 2 * RH;  // rows of a call, at most
  // The state, row-major with the 32-byte groups of row r XORed with r / 8: float (r, c) sits at
  // r*128 + 8((c/8) ^ (r/8 & 15)) + c%8, so the 16 rows of one register-layout access (stride 8
  // rows) hit distinct groups.
  __shared__ __align__(16) float sS[GDN_D * GDN_D];
  __shared__ __align__(16) float sk[GDN_MAXN][GDN_D], sv[GDN_MAXN][GDN_D];  // replayed rows
  __shared__ __align__(16) float qa[MAXN][GDN_D], ka[MAXN][GDN_D], va[MAXN][GDN_D];
  __shared__ __align__(16) float oa[MAXN][GDN_D];
  // gates of the replayed and the new rows: every thread of the loading waves fills a slot of its
  // own (loads that only a branch uses would sink into it, behind the state's)
  __shared__ float sg[LOAD_WAVES * WAVE][2], ga[LOAD_WAVES * WAVE][2], l2p[MAXN][4];
  auto sidx = [](int r, int c) { return r * GDN_D + 8 * ((c >> 3) ^ ((r >> 3) & 15)) + (c & 7); };

  constexpr int NC = 2;  // state columns per lane
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = lane >> 2, col0 = 4 * NC * w + NC * (lane & 3);
  const int j = blockIdx.x, r = Hv / Hk, i = j / r;
  const int C = 2 * Hk * GDN_D + Hv * GDN_D;
  float* Sj = S + (size_t)j * GDN_D * GDN_D;
  const int c = tid & 127;

  float y[RH];           // conv waves: this thread's conv results
  float sz0 = 0.f, sz1 = 0.f, nw0 = 0.f, nw1 = 0.f;  // loading waves: silu(z) and norm weights
  const int hf = w >= 6 ? 1 : 0, w6 = w - 6 * hf, part = w6 >> 1;  // conv: 0 = q, 1 = k, 2 = v
  const int P = ctl[0];
  const int pend = min(max(ctl[1], 0), GDN_MAXN);
  if (w >= CONV_WAVES) {
    // The loading waves move the state and the staged rows to LDS by DMA, one KB (two rows) a
    // load; then they compute the gates and hold the output norm's operands (row w - 12).
    const int lw = w - CONV_WAVES, gt = tid - CONV_WAVES * WAVE;
    const int gtc = min(gt, n - 1), tz = min(lw, n - 1);
    const __bf16 bb = b[(size_t)gtc * ldp + j], ab = a[(size_t)gtc * ldp + j];
    const __bf16 dtb = dt_bias[j], alb = A_log[j];
    const __bf16* zp = z + (size_t)tz * ldp + j * GDN_D + 2 * lane;
    const __bf16 zb0 = zp[0], zb1 = zp[1], nb0 = norm_w[2 * lane], nb1 = norm_w[2 * lane + 1];
    const float2 stg = *reinterpret_cast<const float2*>(st_g + ((size_t)(tid & 7) * Hv + j) * 2);
    __builtin_amdgcn_sched_barrier(0);
    const __amdgpu_buffer_rsrc_t srs = make_rsrc_uniform(Sj, GDN_D * GDN_D * 4);
#pragma unroll
    for (int u = 0; u < GDN_D / 2 / LOAD_WAVES; ++u) {
      const int m = u * LOAD_WAVES + lw;  // rows 2m, 2m + 1
      const uint32_t chunk = (lane & 31) ^ (2 * ((m >> 2) & 15));
      buffer_load16_to_lds<0>(srs, (2 * m + (lane >> 5)) * (GDN_D * 4) + chunk * 16,
                              &sS[2 * m * GDN_D]);
    }
    const uint32_t st_bytes = GDN_MAXN * (uint32_t)Hv * (GDN_D * 4);
    const __amdgpu_buffer_rsrc_t krs = make_rsrc_uniform(st_k, st_bytes);
    const __amdgpu_buffer_rsrc_t vrs = make_rsrc_uniform(st_v, st_bytes);
    static_assert(LOAD_WAVES * 2 == GDN_MAXN, "a staged row pair per loading wave");
    const uint32_t off = ((2 * lw + (lane >> 5)) * Hv + j) * (GDN_D * 4) + (lane & 31) * 16;
    buffer_load16_to_lds<0>(krs, off, sk[2 * lw]);
    buffer_load16_to_lds<0>(vrs, off, sv[2 * lw]);
    __builtin_amdgcn_sched_barrier(0);
    const float2 gv = gate_values(bb, ab, dtb, alb);
    ga[gt][0] = gv.x;
    ga[gt][1] = gv.y;
    sg[gt][0] = stg.x;
    sg[gt][1] = stg.y;
    sz0 = silu_f(bf16_to_f32(zb0));
    sz1 = silu_f(bf16_to_f32(zb1));
    nw0 = bf16_to_f32(nb0);
    nw1 = bf16_to_f32(nb1);
    vmcnt_wait<0>();  // the state and the staged rows are in LDS
  } else if (hf < n) {
    const int ch = part == 0 ? i * GDN_D + c : part == 1 ? (Hk + i) * GDN_D + c
                                                          : 2 * Hk * GDN_D + j * GDN_D + c;
    const uint2 wv = *reinterpret_cast<const uint2*>(conv_w + (size_t)ch * 4);
    constexpr int NX = 2 * RH + 2;
    __bf16 xb[NX];  // positions P + hf - 3 ..
    float xs[NX];
#pragma unroll
    for (int q = 0; q < NX; ++q) xb[q] = conv_input(qkv, ldp, ring, C, P, n, hf + q - 3, ch);
    const float cw[4] = {lo_bf16(wv.x), hi_bf16(wv.x), lo_bf16(wv.y), hi_bf16(wv.y)};
#pragma unroll
    for (int q = 0; q < NX; ++q) xs[q] = conv_value(xb[q], P, hf + q - 3);
    const bool writes_ring = part == 2 || j % r == 0;  // q/k channels are shared by r heads
#pragma unroll
    for (int u = 0; u < RH; ++u) {  // (row hf + 2 may be past n: computed and not used)
      const int t = hf + 2 * u;
      y[u] = conv_silu(cw, xs, 2 * u);
      if (writes_ring && t < n) ring[(size_t)((P + t) & (GDN_RING - 1)) * C + ch] = xb[2 * u + 3];
      if (part == 2) {
        va[t][c] = y[u];
      } else {  // sum of squares of q (w6 = 0, 1) and k (w6 = 2, 3)
        const float ss = wave_sum_fast(y[u] * y[u]);
        if (lane == 0) l2p[t][w6] = ss;
      }
    }
  }
  lds_barrier();  // (the ring's stores need not have arrived)
  float s[8][NC];  // each lane reads (and later writes) only its own elements
#pragma unroll
  for (int rr = 0; rr < 8; ++rr) {
    const float2 v = *reinterpret_cast<const float2*>(&sS[sidx(rg * 8 + rr, col0)]);
    s[rr][0] = v.x;
    s[rr][1] = v.y;
  }

  // Stage this call's v and gates for the next call's replay. Only after the barrier: the staged
  // rows of the previous call (same addresses) have all been read into LDS by then.
  for (int t = tid >> 7; t < n; t += GDN_THREADS / GDN_D)
    st_v[((size_t)t * Hv + j) * GDN_D + c] = va[t][c];
  if (tid < n)
    *reinterpret_cast<float2*>(st_g + ((size_t)tid * Hv + j) * 2) = make_float2(ga[tid][0], ga[tid][1]);

  // Normalise this call's q and k, each thread its own conv results, and stage k for the next
  // call. The rows are read only after the barrier that follows the replay.
  if (w < CONV_WAVES && part < 2 && hf < n) {
    const float sqrt_dk = 11.313708498984761f;  // sqrt(128) rounded to fp32
#pragma unroll
    for (int u = 0; u < RH; ++u) {
      const int t = hf + 2 * u;
      if (t < n) {
        const float inv = 1.0f / sqrtf((l2p[t][2 * part] + l2p[t][2 * part + 1]) + 1e-6f);
        if (part == 0) {
          qa[t][c] = (y[u] * inv) / sqrt_dk;
        } else {
          const float kn = y[u] * inv;
          ka[t][c] = kn;
          st_k[((size_t)t * Hv + j) * GDN_D + c] = kn;
        }
      }
    }
  }

  // ---- 1. replay the rows kept by the previous call, write the committed state back ----
  for (int t = 0; t < pend; ++t) {
    float k[8];
    lds_read8(&sk[t][rg * 8], k);
    const float2 vv = *reinterpret_cast<const float2*>(&sv[t][col0]);
    const float v[NC] = {vv.x, vv.y};
    delta_step(s, k, v, sg[t][0], sg[t][1]);
  }
  if (pend > 0) {
#pragma unroll
    for (int rr = 0; rr < 8; ++rr)
      *reinterpret_cast<float2*>(&sS[sidx(rg * 8 + rr, col0)]) = make_float2(s[rr][0], s[rr][1]);
  }
  lds_barrier();
  if (pend > 0) {  // the copy runs beside the new rows, which do not touch sS
#pragma unroll
    for (int k = 0; k < GDN_D * GDN_D / 4 / GDN_THREADS; ++k) {
      const int f = tid + GDN_THREADS * k;
      reinterpret_cast<F4*>(Sj)[f] = *reinterpret_cast<const F4*>(&sS[sidx(f >> 5, 4 * (f & 31))]);
    }
  }

  // ---- 2. new rows on the register copy ----
  for (int t = 0; t < n; ++t) {
    float k[8], q[8];
    lds_read8(&ka[t][rg * 8], k);
    lds_read8(&qa[t][rg * 8], q);
    const float2 vv = *reinterpret_cast<const float2*>(&va[t][col0]);
    const float v[NC] = {vv.x, vv.y};
    delta_step(s, k, v, ga[t][0], ga[t][1]);
    float o[NC];
    read_out(s, q, o);
    if (rg == 0) *reinterpret_cast<float2*>(&oa[t][col0]) = make_float2(o[0], o[1]);
  }
  lds_barrier();

  // ---- gated RMSNorm: wave 12 + t normalises row t ----
  const int t = w - CONV_WAVES;
  if (t >= 0 && t < n)
    gated_norm_row(oa[t], lane, nw0, nw1, sz0, sz1, eps, out + (size_t)t * ldo + j * GDN_D);
}

}  // namespace qe


using namespace qe;

extern "C" hipError_t qe_gdn_step_n(const void* qkv, const void* z, const void* b, const void* a,
                                    long ldp, void* ring, const void* conv_w, const void* A_log,
                                    const void* dt_bias, const void* norm_w, float* S, float* st_k,
                                    float* st_v, float* st_g, const int* ctl, void* out, long ldo,
                                    int n, int Hk, int Hv, float eps, hipStream_t stream) {
  auto al = [](const void* p, uintptr_t m) { return (reinterpret_cast<uintptr_t>(p) & (m - 1)) == 0; };
  if (!qkv || !z || !b || !a || !ring || !conv_w || !A_log || !dt_bias || !norm_w || !S || !st_k ||
      !st_v || !st_g || !ctl || !out)
    return hipErrorInvalidValue;
  if (n < 1 || n > GDN_MAXN || Hk < 1 || Hv < 1 || Hv % Hk != 0 || Hv > 65535)
    return hipErrorInvalidValue;
  const long C = 2L * Hk * GDN_D + (long)Hv * GDN_D;
  if (C >= (1L << 26) || ldp < C || ldo < (long)Hv * GDN_D) return hipErrorInvalidValue;
  if (!al(S, 16) || !al(st_k, 16) || !al(st_v, 16) || !al(st_g, 8) || !al(conv_w, 8))
    return hipErrorInvalidValue;
  // 5-8 rows: the split kernel and its finish kernel; 1-4 rows: one workgroup per head (below
  // five rows the split's second launch costs more than the spread saves; us per call on MI355X at
  // Hk 16 / Hv 48, n : pending, one workgroup against split: 4:0 8.6 / 9.7, 4:4 10.8 / 11.2, 5:5 12.5 /
  // 12.0, 8:8 16.9 / 14.4). Both paths give the same bits.
  if (n >= GDN_SPLIT_MIN_ROWS)
    return launch_gdn_split(static_cast<const __bf16*>(qkv), static_cast<const __bf16*>(z),
                            static_cast<const __bf16*>(b), static_cast<const __bf16*>(a), ldp,
                            static_cast<__bf16*>(ring), static_cast<const __bf16*>(conv_w),
                            static_cast<const __bf16*>(A_log), static_cast<const __bf16*>(dt_bias),
                            static_cast<const __bf16*>(norm_w), S, st_k, st_v, st_g, ctl,
                            static_cast<__bf16*>(out), ldo, n, Hk, Hv, eps, stream);
  auto kern = n <= 2 ? gdn_step_kernel<1> : gdn_step_kernel<2>;
  kern<<<dim3(Hv), dim3(GDN_THREADS), 0, stream>>>(
      static_cast<const __bf16*>(qkv), static_cast<const __bf16*>(z), static_cast<const __bf16*>(b),
      static_cast<const __bf16*>(a), ldp, static_cast<__bf16*>(ring),
      static_cast<const __bf16*>(conv_w), static_cast<const __bf16*>(A_log),
      static_cast<const __bf16*>(dt_bias), static_cast<const __bf16*>(norm_w), S, st_k, st_v, st_g,
      ctl, static_cast<__bf16*>(out), ldo, n, Hk, Hv, eps);
  return hipGetLastError();
}
