// Chunked-prefill gated attention (the op of attn_prefill.hip) on 32 query columns per wave.
//
//  * A workgroup is four waves, one per SIMD, of 32 columns each: a unit of 128 consecutive columns
//    of one KV head, column = row * (Hq / Hkv) + q head. Consecutive columns are consecutive rows,
//    so the waves of a unit have nearly the same causal length, and any group size works.
//  * S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_32x32x16_bf16: an operand read from LDS feeds
//    32 columns, half the LDS reads per MFMA of 16-column waves.
//  * One wave per SIMD, so the overlap is inside the wave: step j runs S^T of tile j + 1 beside the
//    softmax of tile j, whose second half runs beside the first MFMAs of O^T of tile j. The order is
//    pinned by a scheduling barrier after each MFMA. The loop is bound by the instructions a lone
//    wave can issue: 205 of them a tile (VALU with 32 MFMAs and 16 exponentials, LDS, scalar) take about
//    1,650 clocks against 1,024 of MFMA (counters, 12k caches; at 1.8 to 1.9 GHz under this load).
//  * K and V arrive by LDS DMA in a ring of four stages, one instruction between two MFMAs (issued
//    together they held the wave up: 0.16 us of the 0.98 us a tile then took).
//  * Where the units do not fill the CUs (short chunks on long caches above all), the last U mod W
//    units of a KV head are cut into slices of the cache (slices()); their partials go through a
//    workspace and a second kernel merges them. The slice count depends on the attended length,
//    which only the device knows, so both kernels compute it.
// Measured against the kernels this one replaced, 24 / 4 heads, bf16 cache, us per call (unsplit without a
// workspace): 301 rows on 12,007 positions 420 -> 107 (unsplit 277); 64 on 4,000 151 -> 27 (99); 777 on
// none 42 -> 30; 1,500 on 4,000 196 -> 182; 2,048 rows on 2,048 at 32 / 8 heads 233 -> 198 and at 16 / 2
// 138 -> 114. One unit of an empty cache (9 to 32 rows at group sizes above 1) 11.3 .. 12.0 -> 12.0: the
// epilogue of 32 columns is longer than that of 16.
#include "attn_tile.hpp"
#include "attn_prefill.hpp"

namespace qe {
namespace wide {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) const u32x4_t lds_u32x4;
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) void lds_void;
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
using tile::BN;

constexpr int WAVES = 4;                        // one per SIMD
constexpr int WCOLS = 32;                       // query columns per wave
constexpr int UCOLS = WAVES * WCOLS;            // query columns of a unit (a workgroup)
// P takes two bf16 terms (hi + lo) where a row of a wave is in a block of 16 rows (a multiple of 16 on)
// whose first row attends fewer positions than this: the rows that the balanced kernel, a block per
// wave, gives two terms, and for the rest of the wave no fewer.
constexpr int SPLIT_BELOW = 512, SPLIT_ROWS = 16;
// LDS tiles: rows in pairs of 1024 bytes. K: row 2p + o at 1056 p + 512 o, its 16-byte chunks
// XORed with o, so that 16 rows at one chunk cover all banks; every operand read is one per-lane
// base plus an immediate. V: row 2p + o at 1152 p + 512 o, its 64-byte pieces XORed with o, so that
// 4 rows at one piece cover all banks; two per-lane bases.
constexpr int KPAIR = 2 * HD * 2 + 32, VPAIR = 2 * HD * 2 + 128;
constexpr int KTILE = BN / 2 * KPAIR, STAGE = KTILE + BN / 2 * VPAIR;  // a stage: K tile, V tile
constexpr int STAGES = 4;
// fp8 cache: the codes arrive in rings of four K and four V tiles (rows of 256 bytes); each wave
// converts the rows it loaded into three K and two V tiles of bf16, the latter in the layouts above.
constexpr int TILE8 = BN * HD, VTILE = STAGE - KTILE;
constexpr int V8 = 3 * KTILE, K8RING = V8 + 2 * VTILE, V8RING = K8RING + STAGES * TILE8;
constexpr int RING16 = STAGES * STAGE, RING8 = V8RING + STAGES * TILE8;
constexpr int LOAD_PAIRS = BN / 2 / WAVES;      // row pairs each wave fetches per tile, K and V
constexpr int SLOT_F = UCOLS * HD + WAVES * WAVE * 2;  // floats of a unit's partial

__device__ __forceinline__ f32x16_t mfma32x32x16(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
// x / d for M = floor(2^32 / d) (d = 1: 2^32 - 1): the product is at most one short
__device__ __forceinline__ uint32_t udiv(uint32_t x, uint32_t d, uint32_t M) {
  const uint32_t r = __umulhi(x, M);
  return x - r * d >= d ? r + 1 : r;
}

// What the host knows of a call; the attended lengths depend on pos, which the device reads.
struct Call {
  int T, Hq, Hkv, grp, max_len;
  int U;         // units of a KV head: 128 columns, column = row * grp + q head of the group
  int W;         // workgroups of a KV head that run at once
  int r;         // U % W: the units left when the others fill whole rounds
  int most;      // slices that one of them is cut into at most
  uint32_t grp_m, r_m, Hkv_m;  // for udiv
  float scale_log2, v_scale;
  uint32_t q_flip;
  long ldp, ldo;
};
__device__ __forceinline__ int attended(const Call& s, int pos0, int u) {
  return min(pos0 + min(s.T, (int)udiv((u + 1) * UCOLS - 1, s.grp, s.grp_m) + 1), s.max_len);
}
__device__ __forceinline__ int tiles_of(const Call& s, int pos0, int u) {
  return max(1, (attended(s, pos0, u) + BN - 1) / BN);
}

constexpr float ROUND = 13.f;  // steps of a round of units outside the tile loop
// Estimated time, in tile steps (0.9 us in a full round, bf16 cache), of the last r units (n tiles each)
// cut into S slices: rounds of r S workgroups, and for S > 1 the second kernel, 6 steps and 0.025 for each
// of the slots it reads. Fitted to 24 / 4 heads; checked against 26 calls at 24 / 4, 16 / 2, 4 / 4, 32 / 8, 8 / 1
// and 64 / 8 heads, both caches, 9 to 1,500 rows on 1,000 to 16,000 positions, each timed at up to 20 slice
// counts: the count with the least estimate is within 2% of the fastest one in 13, within 8% in 21; it is
// too large for one or a few units on short prefixes (24% at 100 rows on 2,000 at 4 / 4: 26 slices
// 21.4 us, 12 17.2).
__host__ __device__ inline float slice_cost(int r, int W, int Hkv, int S, float n) {
  const int items = r * S;
  if (S > 1 && items > 2 * W) return 1e30f;
  const float rounds = items <= W ? 1.f : items <= 2 * W ? 2.f : 3.f;
  return rounds * (n / (float)S + ROUND) + (S > 1 ? 6.f + 0.025f * (float)(items * Hkv) : 0.f);
}
// Slices of the cache that the last r units are cut into: the count with the least estimated time.
__device__ __forceinline__ int slices(const Call& s, int pos0, int lane) {
  const float n = (float)tiles_of(s, pos0, s.r - 1);
  const float cost = lane < s.most ? slice_cost(s.r, s.W, s.Hkv, lane + 1, n) : 2e30f;
  float m = fminf(cost, dpp<0xB1>(cost));
  m = fminf(m, dpp<0x4E>(m));
  m = fminf(m, dpp<0x1B>(dpp<0x141>(m)));
  m = fminf(m, dpp<0x128>(m));
  m = -group4_max(-m);
  return __builtin_ctzll(__ballot(cost == m)) + 1;
}

// This wave's LDS-DMA loads of one K or V tile: rows 8w .. 8w+7, a pair of rows per instruction
// (i = 0..3). rs starts at row 8w of the tile; dst is the LDS byte address of that row; off the
// lane's byte offset in a pair (the immediate offset counts for the LDS address too).
template <int PAIR>
__device__ __forceinline__ void load_pair(__amdgpu_buffer_rsrc_t rs, uint32_t dst, uint32_t off, int i) {
  if (i == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(uintptr_t)dst, 16, off, 0, 0, 0);
  if (i == 1) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(uintptr_t)(dst + PAIR - 1024), 16, off, 0, 1024, 0);
  if (i == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(uintptr_t)(dst + 2 * (PAIR - 1024)), 16, off, 0, 2048, 0);
  if (i == 3) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(uintptr_t)(dst + 3 * (PAIR - 1024)), 16, off, 0, 3072, 0);
}
template <bool KV8>
struct Ring {
  __amdgpu_buffer_rsrc_t krs, vrs;  // this KV head's rows up to the last one needed; past it zeros
  uint32_t ko, vo;                  // this lane's byte offset in the wave's first rows of tile 0
  uint32_t at[STAGES];  // LDS byte addresses: bf16 cache, the stages of tiles j .. j + 3; fp8 cache,
                        // the K tiles j, j + 1, j + 2 (at[3]: V tile j + 1)
  uint32_t vt;          // V tile j
  uint32_t kw, vw;      // this wave's rows: in a stage; fp8 cache, in the rings of codes
  // a load instruction (i) of K or V tile j
  template <bool V>
  __device__ __forceinline__ void load(int j, int i) const {
    if constexpr (KV8) {
      const uint32_t off = (V ? vo : ko) + (uint32_t)j * TILE8, dst = (V ? vw : kw) + (j & 3) * TILE8;
      const __amdgpu_buffer_rsrc_t rs = V ? vrs : krs;
      if (i == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(uintptr_t)dst, 16, off, 0, 0, 0);
      if (i == 1) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void*)(uintptr_t)dst, 16, off, 0, 1024, 0);
    } else {
      const uint32_t off = (V ? vo : ko) + (uint32_t)j * (BN * HD * 2);
      const uint32_t stage = at[V ? 3 : 0];  // V(j + 3) over V(j - 1), K(j + 4) over K(j)
      load_pair<V ? VPAIR : KPAIR>(V ? vrs : krs, stage + (V ? vw : kw), off, i);
    }
  }
  __device__ __forceinline__ void next() {
    if constexpr (KV8) {
      uint32_t t = at[0];
      at[0] = at[1], at[1] = at[2], at[2] = t;
      t = vt, vt = at[3], at[3] = t;
    } else {
      const uint32_t t = at[0];
      at[0] = at[1], at[1] = at[2], at[2] = at[3], at[3] = t;
      vt = at[0] + KTILE;
    }
  }
};

// Conversion of this wave's 8 rows of an fp8 tile: lane -> 8 codes of row 2t + (lane >> 5), t = 0..3.
struct Convert {
  uint32_t src, kdst, vdst;  // per lane: in a tile of codes, in a K tile, in a V tile
  u32x2_t k[4], v[4];
  __device__ __forceinline__ void init(int w, int lane) {
    const uint32_t o = lane >> 5, q = lane & 31;
    src = (8 * w + o) * HD + 8 * q;
    kdst = 4 * w * KPAIR + o * (HD * 2) + 16 * (q ^ o);
    vdst = 4 * w * VPAIR + o * (HD * 2) + 16 * (q ^ (4 * o));
  }
  __device__ __forceinline__ u32x2_t read(uint32_t tile, int t) const {
    typedef __attribute__((address_space(3))) const u32x2_t lds_cu32x2;
    return *(lds_cu32x2*)(uintptr_t)(tile + src + 2 * HD * t);
  }
  template <bool V>
  __device__ __forceinline__ void write(uint32_t tile, int t, u32x2_t x) const {
    typedef __attribute__((address_space(3))) u32x4_t lds_wu32x4;
    *(lds_wu32x4*)(uintptr_t)(tile + (V ? vdst + VPAIR * t : kdst + KPAIR * t)) = fp8x8_to_bf16x8(x);
  }
};

// bf16(sigmoid_f32(x)) of a pair of bf16 x, the same bits for all 65,536 of them (checked on MI355X), by
// the hardware exponential and reciprocal. The reciprocal flushes subnormal results, so it is taken of
// (1 + e) 2^-24 and scaled back: gates below -87.3 are subnormal, not 0.
__device__ __forceinline__ uint32_t gates(uint32_t x) {
  constexpr float s = 0x1p-24f;
  float y[2] = {lo_bf16(x), hi_bf16(x)};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float e = __builtin_amdgcn_exp2f(-1.4426950408889634f * y[i]);
    y[i] = __builtin_amdgcn_rcpf(__builtin_fmaf(e, s, s)) * s;
  }
  return pack_bf16x2(y[0], y[1]);
}
// bf16 products of two pairs
__device__ __forceinline__ uint32_t mul_bf16x2(uint32_t a, uint32_t b) {
  return pack_bf16x2(lo_bf16(a) * lo_bf16(b), hi_bf16(a) * hi_bf16(b));
}

// acc / L to within 2^-22 of a half ulp of the correctly rounded quotient, as two products: 1 / L is
// hi + lo with lo > 0, so that infinities and NaN come out as a division gives them.
struct Quotient {
  float hi, lo;
  __device__ __forceinline__ explicit Quotient(float L) {
    const float r = 1.f / L;
    hi = r > 0.f ? __uint_as_float(__float_as_uint(r) - 1) : r;
    lo = fmaxf(__builtin_fmaf(-L, hi, 1.f) * r, 1.17549435e-38f);
  }
  __device__ __forceinline__ float operator()(float acc) const { return __builtin_fmaf(acc, hi, acc * lo); }
};

struct State {
  float m, l;
  f32x16_t acc[8];  // acc[i][r] = O^T[32i + 8(r>>2) + 4h + (r&3)][column c]
};
struct Probs {
  u32x4_t hi[2], lo[2];
};

__device__ __forceinline__ bf16x8_t k_read(uint32_t k0, int ks) {
  return as_bf16x8(*(lds_u32x4*)(uintptr_t)(k0 + 32 * ks));
}
__device__ __forceinline__ uint32_t k_base(uint32_t kt, int lane) {
  const int r = lane & 31, h = lane >> 5;
  return kt + (r >> 1) * KPAIR + (r & 1) * (HD * 2) + 16 * (h ^ (r & 1));
}

// One step of the softmax of a tile, spread over the MFMAs of the next tile's S^T (part 0..15).
// s: raw scores; position of s[e]: p0 + 8(e>>2) + 4h + (e&3).
template <bool MASK, bool SPLIT>
struct Softmax {
  f32x16_t s;
  float t, corr, msub, sum[2];
  bool moved;
  __device__ __forceinline__ void exps(int e, float scale) {
    float x = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], scale, -msub));
    asm volatile("" : "+v"(x));  // evaluated here, beside the MFMAs
    s[e] = x;
    sum[e & 1] += x;
  }
  __device__ __forceinline__ void pack(int d, Probs& p) {
    p.hi[d >> 2][d & 3] = pack_bf16x2(s[2 * d], s[2 * d + 1]);
    if constexpr (SPLIT)
      p.lo[d >> 2][d & 3] = pack_bf16x2(s[2 * d] - lo_bf16(p.hi[d >> 2][d & 3]),
                                        s[2 * d + 1] - hi_bf16(p.hi[d >> 2][d & 3]));
  }
  __device__ __forceinline__ void part(int k, int left, float scale, State& st, Probs& p) {
    // left: Lcol - p0 - 4h
    if (k < 4) {
      if constexpr (MASK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s[4 * k + i] = 8 * k + i < left ? s[4 * k + i] : -INFINITY;
      }
      const float a = fmaxf(fmaxf(s[4 * k], s[4 * k + 1]), s[4 * k + 2]);
      t = k ? fmaxf(fmaxf(t, a), s[4 * k + 3]) : fmaxf(a, s[4 * k + 3]);
    } else if (k == 4) {
      t = xor32_pair(t, false) * scale;
    } else if (k == 5) {
      moved = false;
      corr = 1.f;
      if (t > st.m + tile::LAZY_TAU) {
        if (st.m != -INFINITY) {
          corr = __builtin_amdgcn_exp2f(st.m - t);
          moved = true;
        }
        st.m = t;
      }
      msub = st.m == -INFINITY ? 0.f : st.m;
      sum[0] = sum[1] = 0.f;
    } else if (k < 14) {
      exps(k - 6, scale);
      if ((k & 1) && k > 6) pack((k - 7) / 2, p);
    }
  }
  // the other half of the tile, spread over the first 8 MFMAs of O^T (part 0..7)
  __device__ __forceinline__ void late(int k, float scale, State& st, Probs& p) {
    exps(8 + k, scale);
    if (k & 1) pack(4 + k / 2, p);
    if (k == 7) st.l = st.l * corr + (sum[0] + sum[1]);
  }
};

// V^T operand reads of a tile: operand k = M-tile k % 8 of k-step k / 8.
struct VRead {
  lds_char* b[2];
  // row 16s + 8u + 4h + x of the tile, dims 32i + 16 ((lane >> 4) & 1) + 4 (lane & 3) .. +3; piece
  // i of the row is at i ^ (x & 1)
  __device__ __forceinline__ VRead(lds_char* __restrict__ vt, int lane) {
    const int x = (lane >> 2) & 3, o = x & 1;
    lds_char* v0 = vt + (2 * (lane >> 5) + (x >> 1)) * VPAIR + o * (HD * 2) +
                   32 * ((lane >> 4) & 1) + 8 * (lane & 3);
    b[0] = v0 + 64 * o;
    b[1] = v0 + 64 * (1 - o);
  }
  __device__ __forceinline__ bf16x8_t operator()(int k) const {
    const int i = k & 7, s = k >> 3;
    lds_char* a = b[i & 1] + 64 * (i & 6) + 8 * s * VPAIR;
    const u32x2_t x = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)a));
    const u32x2_t y = __builtin_bit_cast(
        u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(a + 4 * VPAIR)));
    return as_bf16x8(u32x4_t{x[0], x[1], y[0], y[1]});
  }
};

constexpr int LEAD = 6;  // operand reads ahead of the MFMAs

// Step j: S^T of tile j + 1 beside the first half of tile j's softmax, then O^T += V^T P^T of tile
// j beside the second half. The operands of two MFMAs in a row are waited for together: the later
// read's MFMA goes first.
template <bool KV8, bool MASK, bool SPLIT>
__device__ __forceinline__ void step(lds_char* __restrict__ vt, int j, const Ring<KV8>& rg, Convert& cv,
                                     uint32_t base, int Lcol, int lane, const bf16x8_t (&qb)[16],
                                     float scale, bf16x8_t (&kop)[LEAD], f32x16_t& sc, State& st) {
  Softmax<MASK, SPLIT> sm;
  sm.s = sc;
  Probs p;
  const int left = Lcol - j * BN - 4 * (lane >> 5);
  const uint32_t k0 = k_base(rg.at[1], lane), k1 = k_base(rg.at[2], lane);
  const VRead vr(vt, lane);
  bf16x8_t ko[16 + LEAD], vo[16];
#pragma unroll
  for (int i = 0; i < LEAD; ++i) ko[i] = kop[i];
  f32x16_t n = (f32x16_t)(0.f);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int ks = i ^ 1;
    n = mfma32x32x16(ko[ks], qb[ks], n);
    if (i & 1) {
#pragma unroll
      for (int r = i + LEAD - 1; r < i + LEAD + 1; ++r) {
        if (r < 16)
          ko[r] = k_read(k0, r);
        else
          vo[r - 16] = vr(r - 16);
      }
    } else if (i < (KV8 ? 4 : 8)) {
      rg.template load<false>(j + (KV8 ? 6 : 4), i / 2);
    }
    if (KV8 && i >= 14) {  // the codes of K(j + 3), V(j + 1)
#pragma unroll
      for (int t = 2 * (i - 14); t < 2 * (i - 14) + 2; ++t) {
        cv.k[t] = cv.read(base + K8RING + ((j + 3) & 3) * TILE8, t);
        cv.v[t] = cv.read(base + V8RING + ((j + 1) & 3) * TILE8, t);
      }
    }
    sm.part(i, left, scale, st, p);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (__any(sm.moved)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) st.acc[i] *= sm.corr;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int k = i ^ 1;
    st.acc[k & 7] = mfma32x32x16(vo[k], as_bf16x8(p.hi[k >> 3]), st.acc[k & 7]);
    if constexpr (SPLIT) st.acc[k & 7] = mfma32x32x16(vo[k], as_bf16x8(p.lo[k >> 3]), st.acc[k & 7]);
    if (i & 1) {
#pragma unroll
      for (int r = i + LEAD - 1; r < i + LEAD + 1; ++r) {
        if (r < 16)
          vo[r] = vr(r);
        else
          kop[r - 16] = k_read(k1, r - 16);
      }
    } else if (i >= (KV8 ? 12 : 8)) {
      rg.template load<true>(j + (KV8 ? 4 : 3), i / 2 - (KV8 ? 6 : 4));
    }
    if (i < 8) sm.late(i, scale, st, p);
    if (KV8 && i >= 8 && i < 12) cv.template write<false>(rg.at[0], i - 8, cv.k[i - 8]);
    if (KV8 && i >= 12) cv.template write<true>(rg.at[3], i - 12, cv.v[i - 12]);
    __builtin_amdgcn_sched_barrier(0);
  }
  sc = n;
}

// Barrier of step j. bf16 cache: it orders the loads of V(j) and K(j + 2) before their reads and
// frees the stages of K(j) and V(j - 1), which K(j + 4) and V(j + 3) refill (loads in flight at that
// point: V(j + 1), K(j + 3), V(j + 2)). fp8 cache: it orders the bf16 tiles V(j) and K(j + 2) before
// their reads and frees those of K(j) and V(j - 1), which K(j + 3) and V(j + 1) refill; this wave's
// codes of those two have landed (in flight: K and V of two steps), and the codes of K(j + 2) and
// V(j), which it has converted, are replaced by those of K(j + 6) and V(j + 4).
template <bool KV8>
__device__ __forceinline__ void step_barrier() {
  vmcnt_wait<KV8 ? 8 : 12>();
  if constexpr (KV8)
    lds_barrier();
  else
    barrier_no_drain();
}
// Tiles [j0, j1): `sc` holds the scores of tile j at the start of step j, `kop` the first operands
// of tile j + 1.
template <bool KV8, bool MASK, bool SPLIT>
__device__ __forceinline__ void run_tiles(int j0, int j1, Ring<KV8>& rg, Convert& cv, uint32_t base,
                                          int Lcol, int lane, bf16x8_t (&qb)[16], float scale,
                                          bf16x8_t (&kop)[LEAD], f32x16_t& sc, State& st) {
  for (int j = j0; j < j1; ++j) {
    step_barrier<KV8>();
    // q in accumulation registers, so that the rest fits the 256 VGPRs without copies
#pragma unroll
    for (int i = 0; i < 16; ++i) asm volatile("" : "+a"(qb[i]));
    step<KV8, MASK, SPLIT>((lds_char*)(uintptr_t)rg.vt, j, rg, cv, base, Lcol, lane, qb, scale, kop, sc, st);
    rg.next();
  }
}

constexpr int ROW_B = HD * 2 + 16;  // LDS bytes of a column's output in the epilogue

template <bool KV8>
__global__ void __launch_bounds__(WAVES * WAVE)
attn_prefill_wide_kernel(const __bf16* __restrict__ q, const void* __restrict__ kc_,
                         const void* __restrict__ vc_, const int* __restrict__ pos_ptr,
                         const __bf16* __restrict__ qg, __bf16* __restrict__ out,
                         float* __restrict__ ws, Call s) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int pos0 = pos_ptr[0];
  const int item = udiv(blockIdx.x, s.Hkv, s.Hkv_m), g = blockIdx.x - item * s.Hkv;
  __shared__ __attribute__((aligned(256))) u32x4_t lds[(KV8 ? RING8 : RING16) / 16];

  // whole units first, the longest ahead; then the slices of the last r units
  int u = s.U - 1 - item, k = 0, S = 1;
  if (u < s.r) {
    if (ws) S = slices(s, pos0, lane);
    const int i = s.r - 1 - u;
    k = udiv(i, s.r, s.r_m);
    u = s.r - 1 - (i - k * s.r);
    if (k >= S) return;
  }
  const int n = tiles_of(s, pos0, u);
  const int J0 = n * k / S, J1 = n * (k + 1) / S;
  const int c = lane & 31, h = lane >> 5;
  const int c0 = u * UCOLS + w * WCOLS;  // this wave's columns
  const int r0 = udiv(c0, s.grp, s.grp_m);
  const int lc = c0 - r0 * s.grp + c, dr = udiv(lc, s.grp, s.grp_m);
  const int row = r0 + dr, hd = g * s.grp + lc - dr * s.grp;
  const bool wlive = r0 < s.T, live = row < s.T;
  constexpr int ROW = KV8 ? HD : HD * 2;  // bytes of a cache row
  const size_t head = (size_t)g * s.max_len * ROW;
  const uint32_t end = (uint32_t)min(max(attended(s, pos0, u), 0), J1 * BN) * ROW;
  const uint32_t base = lds_byte_uniform(lds);
  Ring<KV8> rg;
  Convert cv;
  rg.krs = make_rsrc_uniform(static_cast<const char*>(kc_) + head, end);
  rg.vrs = make_rsrc_uniform(static_cast<const char*>(vc_) + head, end);
  if constexpr (KV8) {
    rg.ko = rg.vo = (8 * w + (lane >> 4)) * HD + (lane & 15) * 16;
    rg.at[0] = base, rg.at[1] = base + KTILE, rg.at[2] = base + 2 * KTILE;
    rg.vt = base + V8, rg.at[3] = base + V8 + VTILE;
    rg.kw = base + K8RING + 8 * w * HD, rg.vw = base + V8RING + 8 * w * HD;
    cv.init(w, lane);
  } else {
    const uint32_t o = lane >> 5, first = (2 * LOAD_PAIRS * w + o) * (HD * 2);
    rg.ko = first + ((lane & 31) ^ o) * 16;
    rg.vo = first + ((lane & 31) ^ (4 * o)) * 16;
    rg.kw = LOAD_PAIRS * w * KPAIR;
    rg.vw = KTILE + LOAD_PAIRS * w * VPAIR;
  }
  // K or V tile j of the first ones (bf16 cache: stage j - J0)
  auto load_all = [&](auto v, int j) __attribute__((always_inline)) {
    constexpr bool V = decltype(v)::value;
    if constexpr (!KV8) rg.at[V ? 3 : 0] = base + (j - J0) * STAGE;
#pragma unroll
    for (int i = 0; i < (KV8 ? 2 : 4); ++i) rg.template load<V>(j, i);
  };
  using K_ = std::integral_constant<bool, false>;
  using V_ = std::integral_constant<bool, true>;
  load_all(K_{}, J0);
  bf16x8_t qb[16];
  const u32x4_t* src = reinterpret_cast<const u32x4_t*>(q + ((size_t)min(row, s.T - 1) * s.Hq + hd) * HD);
#pragma unroll
  for (int ks = 0; ks < 16; ++ks) qb[ks] = as_bf16x8(src[2 * ks + h]);
  load_all(K_{}, J0 + 1);
  if constexpr (KV8) load_all(K_{}, J0 + 2);
  load_all(V_{}, J0);

  const int Lcol = live ? min(pos0 + row + 1, s.max_len) : 0;
  const int Lmin = min(pos0 + r0 + 1, s.max_len);
  // tiles below the wave's shortest row need no mask; a short range takes one loop
  const int Lwave = min(pos0 + (int)udiv(c0 + WCOLS - 1, s.grp, s.grp_m) + 1, min(pos0 + s.T, s.max_len));
  const int je = wlive ? max(J0, min(J1, (max(Lwave, 0) + BN - 1) / BN)) : J0;  // tiles past its rows
  const int jm = je - J0 < 3 ? J0 : max(J0, min(je, max(Lmin, 0) / BN));

  State st;
  st.m = -INFINITY;
  st.l = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) st.acc[i] = (f32x16_t)(0.f);
  if constexpr (KV8) {
    load_all(K_{}, J0 + 3);
    load_all(V_{}, J0 + 1);
    vmcnt_wait<4>();  // K(J0) .. K(J0 + 2), V(J0) (and q)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        if (J0 + i < J1)  // the scores of a tile past the last one are not used
          cv.template write<false>(rg.at[i], t, cv.read(base + K8RING + ((J0 + i) & 3) * TILE8, t));
      cv.template write<true>(rg.vt, t, cv.read(base + V8RING + (J0 & 3) * TILE8, t));
    }
    load_all(K_{}, J0 + 4);
    load_all(V_{}, J0 + 2);
    load_all(K_{}, J0 + 5);
    load_all(V_{}, J0 + 3);
    lds_barrier();
  } else {
    vmcnt_wait<8>();  // K(J0) (and q)
    barrier_no_drain();
    // the rest of the ring's first tiles, beside the first scores
    load_all(K_{}, J0 + 2);
    load_all(V_{}, J0 + 1);
    load_all(K_{}, J0 + 3);
    load_all(V_{}, J0 + 2);
#pragma unroll
    for (int i = 0; i < STAGES; ++i) rg.at[i] = base + i * STAGE;
    rg.vt = base + KTILE;
  }
  if (je > J0) {
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) qb[ks] = as_bf16x8(__builtin_bit_cast(u32x4_t, qb[ks]) ^ s.q_flip);
    f32x16_t sc = (f32x16_t)(0.f);
    const uint32_t k0 = k_base(rg.at[0], lane), k1 = k_base(rg.at[1], lane);
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) sc = mfma32x32x16(k_read(k0, ks), qb[ks], sc);
    if constexpr (!KV8) {
      vmcnt_wait<20>();  // K(J0 + 1)
      barrier_no_drain();
    }
    bf16x8_t kop[LEAD];
#pragma unroll
    for (int i = 0; i < LEAD; ++i) kop[i] = k_read(k1, i);
    auto run = [&](auto mk, auto sp, int j0, int j1) __attribute__((always_inline)) {
      run_tiles<KV8, decltype(mk)::value, decltype(sp)::value>(j0, j1, rg, cv, base, Lcol, lane, qb,
                                                               s.scale_log2, kop, sc, st);
    };
    if (min(pos0 + (r0 & -SPLIT_ROWS) + 1, s.max_len) < SPLIT_BELOW) {
      run(K_{}, V_{}, J0, jm);
      run(V_{}, V_{}, jm, je);
    } else {
      run(K_{}, K_{}, J0, jm);
      run(V_{}, K_{}, jm, je);
    }
  } else if constexpr (!KV8) {
    vmcnt_wait<20>();
    barrier_no_drain();
  }
  for (int j = je; j < J1; ++j) {  // past its rows a wave only loads (and converts)
    step_barrier<KV8>();
    if constexpr (KV8) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        cv.template write<false>(rg.at[0], t, cv.read(base + K8RING + ((j + 3) & 3) * TILE8, t));
        cv.template write<true>(rg.at[3], t, cv.read(base + V8RING + ((j + 1) & 3) * TILE8, t));
      }
    }
#pragma unroll
    for (int i = 0; i < (KV8 ? 2 : 4); ++i) rg.template load<false>(j + (KV8 ? 6 : 4), i);
#pragma unroll
    for (int i = 0; i < (KV8 ? 2 : 4); ++i) rg.template load<true>(j + (KV8 ? 4 : 3), i);
    rg.next();
  }
  vmcnt_wait<0>();  // no LDS DMA may still target this workgroup's LDS
  const float L = xor32_pair(st.l, true);
  if (S > 1) {
    if (!wlive) return;
    float* slot = ws + ((size_t)g * s.r * s.most + u * S + k) * SLOT_F;
    f32x4_t* po = reinterpret_cast<f32x4_t*>(slot) + w * 32 * WAVE + lane;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        po[(i * 4 + b) * WAVE] = f32x4_t{st.acc[i][4 * b], st.acc[i][4 * b + 1],
                                         st.acc[i][4 * b + 2], st.acc[i][4 * b + 3]};
    float* ml = slot + UCOLS * HD + (w * WAVE + lane) * 2;
    ml[0] = st.m;
    ml[1] = L;
    return;
  }
  // O / l as bf16 and the gate rows to LDS (the ring is idle once every wave is here), then whole
  // rows: a short loop instead of one unrolled over the accumulators, whose code would be fetched cold
  lds_barrier();
  if (!wlive) return;
  const uint32_t ob = base + w * (WCOLS * ROW_B), gt = base + WAVES * WCOLS * ROW_B + w * (WCOLS * HD * 2);
  const int pairs = (min(WCOLS, s.T * s.grp - c0) + 1) / 2;  // of live columns
  // A lane takes every second column; its place in the gate and output rows moves on by additions. With
  // that, the next pair's LDS reads ahead of this pair's arithmetic and no pairs of dead columns, 16 rows
  // of an empty cache at 16 / 2 heads take 12.0 us (12.7 with divisions for every column), 9 rows at
  // 8 / 8 7.6 (8.8), 2,048 rows on 2,048 at 32 / 8 198 (202).
  const int drow = udiv(2, s.grp, s.grp_m), dhd = 2 - drow * s.grp;
  const int l0 = c0 - r0 * s.grp + h, d0 = udiv(l0, s.grp, s.grp_m);
  struct Walk {
    int row, hd;  // row, q head of the group
    long at;      // element
  };
  const auto next = [&](Walk& k, long ld, int width) __attribute__((always_inline)) {
    k.row += drow, k.hd += dhd, k.at += drow * ld + dhd * width;
    if (k.hd >= s.grp) k.hd -= s.grp, ++k.row, k.at += ld - s.grp * width;
  };
  const Walk k0{r0 + d0, l0 - d0 * s.grp, 0};
  const __bf16* gq = qg + (size_t)(g * s.grp) * 2 * HD + HD + 8 * c;
  Walk kg = k0;
  kg.at = kg.row * s.ldp + kg.hd * (2 * HD);
#pragma unroll 4
  for (int t = 0; t < pairs; ++t) {
    const __bf16* src = gq + (kg.row < s.T ? kg.at : r0 * s.ldp);
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                     (lds_void*)(uintptr_t)(gt + 1024 * t), 16, 0, 0);
    next(kg, s.ldp, 2 * HD);
  }
  const Quotient by(L);
  const auto o2 = [&](int i, int r) __attribute__((always_inline)) {  // two values of O as bf16
    float a = by(st.acc[i][r]), b = by(st.acc[i][r + 1]);
    if constexpr (KV8) a *= s.v_scale, b *= s.v_scale;
    return pack_bf16x2(a, b);
  };
  typedef __attribute__((address_space(3))) u32x2_t lds_u32x2;
  const uint32_t wr = ob + c * ROW_B + 8 * h;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int b = 0; b < 4; ++b)
      *(lds_u32x2*)(uintptr_t)(wr + 64 * i + 16 * b) =
          u32x2_t{o2(i, 4 * b), o2(i, 4 * b + 2)};
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  vmcnt_wait<0>();
  Walk ko = k0;
  ko.at = ko.row * s.ldo + ko.hd * HD;
  __bf16* oq = out + (size_t)(g * s.grp) * HD + 8 * c;
  const auto read = [&](int t, u32x4_t (&x)[2]) __attribute__((always_inline)) {
    x[0] = *(lds_u32x4*)(uintptr_t)(ob + (2 * t + h) * ROW_B + 16 * c);
    x[1] = *(lds_u32x4*)(uintptr_t)(gt + 1024 * t + 16 * lane);
  };
  u32x4_t x[2], y[2];
  read(0, x);
#pragma unroll 2
  for (int t = 0; t < pairs; ++t) {
    read(min(t + 1, pairs - 1), y);  // one pair ahead
    u32x4_t r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = mul_bf16x2(x[0][i], gates(x[1][i]));
    asm volatile("" : "+v"(r));  // (not sunk into the branch)
    if (ko.row < s.T) *reinterpret_cast<u32x4_t*>(oq + ko.at) = r;
    next(ko, s.ldo, HD);
    x[0] = y[0], x[1] = y[1];
  }
}

// Merges the partials of the units' slices. One wave per (unit, wave of the unit, 16 dims).
constexpr int CW = 4;  // waves per workgroup
__global__ void __launch_bounds__(CW * WAVE)
attn_prefill_wide_combine(const int* __restrict__ pos_ptr, const __bf16* __restrict__ qg,
                          __bf16* __restrict__ out, const float* __restrict__ ws, Call s) {
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int g = blockIdx.y, u = blockIdx.x / WAVES, w = blockIdx.x % WAVES;
  const int ib = blockIdx.z * CW + threadIdx.x / WAVE;  // dims 16 ib ..
  const int S = slices(s, pos_ptr[0], lane);
  if (S == 1) return;
  const int c0 = u * UCOLS + w * WCOLS, r0 = udiv(c0, s.grp, s.grp_m);
  if (r0 >= s.T) return;
  const int lc = c0 - r0 * s.grp + c, dr = udiv(lc, s.grp, s.grp_m);
  const int row = r0 + dr, hd = g * s.grp + lc - dr * s.grp;
  const float* slots = ws + ((size_t)g * s.r * s.most + u * S) * SLOT_F;
  const float* ml = slots + UCOLS * HD + (w * WAVE + lane) * 2;
  const f32x4_t* po = reinterpret_cast<const f32x4_t*>(slots) + (w * 32 + ib * 2) * WAVE + lane;
  const int d0 = 16 * ib + 8 * h;
  const u32x4_t gb = *reinterpret_cast<const u32x4_t*>(qg + (size_t)min(row, s.T - 1) * s.ldp + (size_t)hd * 2 * HD + HD + d0);
  float m = -INFINITY, L = 0.f;
  f32x4_t o[2] = {(f32x4_t)(0.f), (f32x4_t)(0.f)};
  constexpr int B = 4;  // slices in flight
  for (int k = 0; k < S; k += B) {
    float mk[B], lk[B];
    f32x4_t x[B], y[B];
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const size_t at = (size_t)min(k + i, S - 1) * SLOT_F;
      mk[i] = ml[at];
      lk[i] = ml[at + 1];
      x[i] = po[at / 4];
      y[i] = po[at / 4 + WAVE];
    }
    float mn = m;
#pragma unroll
    for (int i = 0; i < B; ++i) mn = fmaxf(mn, k + i < S ? mk[i] : -INFINITY);
    const float c0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn);
    L *= c0;
    o[0] *= c0;
    o[1] *= c0;
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const bool in = k + i < S && mk[i] != -INFINITY;
      const float e = in ? __builtin_amdgcn_exp2f(mk[i] - mn) : 0.f;
      L += lk[i] * e;
      o[0] += x[i] * e;
      o[1] += y[i] * e;
    }
    m = mn;
  }
  const Quotient by(L);
  uint32_t x[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    x[k] = pack_bf16x2(by(o[k >> 1][2 * (k & 1)]) * s.v_scale, by(o[k >> 1][2 * (k & 1) + 1]) * s.v_scale);
  // both halves of the column's 8-dim block: lane half h gets block h
  const auto e0 = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
  const auto e1 = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
  const uint32_t ov[4] = {e0[0], e1[0], e0[1], e1[1]};
  u32x4_t ob;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    ob[k] = mul_bf16x2(ov[k], gates(gb[k]));
  if (row < s.T)
    *reinterpret_cast<u32x4_t*>(out + (size_t)row * s.ldo + (size_t)hd * HD + d0) = ob;
}

}  // namespace wide
}  // namespace qe

using namespace qe;

// floor(2^32 / d) for udiv
static uint32_t magic(int d) { return d == 1 ? 0xffffffffu : (uint32_t)((1ull << 32) / d); }

// Slices of the last r units at n tiles each (the kernels' slices()).
static int fewest_steps(const wide::Call& s, float n) {
  int best = 1;
  float least = wide::slice_cost(s.r, s.W, s.Hkv, 1, n);
  for (int S = 2; s.r && S <= WAVE && s.r * S <= 2 * s.W; ++S) {
    const float cost = wide::slice_cost(s.r, s.W, s.Hkv, S, n);
    if (cost < least) least = cost, best = S;
  }
  return best;
}
static wide::Call units(int T, int Hq, int Hkv) {
  wide::Call s{};
  s.T = T, s.Hq = Hq, s.Hkv = Hkv, s.grp = Hq / Hkv;
  s.U = (int)(((long)T * s.grp + wide::UCOLS - 1) / wide::UCOLS);
  s.W = compute_units() / Hkv > 0 ? compute_units() / Hkv : 1;
  s.r = s.U % s.W;
  return s;
}
// (`most`: the slices at the longest prefix the cache can hold; a shorter one takes no more)
static wide::Call plan(int T, int Hq, int Hkv, int max_len) {
  wide::Call s = units(T, Hq, Hkv);
  s.max_len = max_len;
  s.most = fewest_steps(s, (float)(((long)max_len + tile::BN - 1) / tile::BN));
  s.grp_m = magic(s.grp), s.Hkv_m = magic(Hkv), s.r_m = magic(s.r ? s.r : 1);
  return s;
}

bool qe::prefill_wide_valid(int T, int Hq, int Hkv) {
  const wide::Call s = units(T, Hq, Hkv);
  return ((long)s.U + 2 * s.W) * Hkv <= 0x7fffffffL && (long)T * s.grp < 0x7fffffffL - wide::UCOLS;
}

// Whole rounds run their units' average length; the last r units are the shortest ones, alone on the
// CUs (faster tiles) or in slices (9 steps are the fp8 cache's first tiles, converted per slice); no call
// ends before its longest unit.
float qe::prefill_wide_steps(int T, int Hq, int Hkv, int max_len, bool ws) {
  const wide::Call s = units(T, Hq, Hkv);
  const float pos = (float)(max_len > T ? max_len - T : 0), rows = (float)T, part = (float)s.r / (float)s.U;
  float steps = (float)(s.U / s.W) * ((pos + rows * (1.f + part) / 2) / tile::BN + wide::ROUND);
  if (s.r) {
    const float n = (pos + rows * part) / tile::BN;
    const int S = ws ? fewest_steps(s, n) : 1;
    steps += S > 1 ? wide::slice_cost(s.r, s.W, s.Hkv, S, n) + 9.f
                   : (n + wide::ROUND) * (0.8f + 0.2f * (float)s.r / (float)s.W);
  }
  const float longest = (pos + rows) / tile::BN + wide::ROUND;
  return steps > longest ? steps : longest;
}

size_t qe::prefill_wide_ws_bytes(int T, int Hq, int Hkv, int max_len) {
  const wide::Call s = plan(T, Hq, Hkv, max_len);
  return s.most > 1 ? (size_t)Hkv * s.r * s.most * wide::SLOT_F * sizeof(float) : 0;
}
size_t qe::prefill_wide_ws_most(int Hkv) {
  return (size_t)Hkv * 2 * units(1, Hkv, Hkv).W * wide::SLOT_F * sizeof(float);
}

hipError_t qe::launch_prefill_wide(const void* q, const void* kc, const void* vc, const int* pos,
                                   const void* qg, long ldp, void* out, long ldo, int T, int Hq,
                                   int Hkv, int max_len, float scale, bool kv8, float v_scale,
                                   float* ws, hipStream_t stream) {
  wide::Call s = plan(T, Hq, Hkv, max_len);
  // a negative scale is the positive one on negated q; 0 as the least normal, so that masked scores
  // (-inf) stay -inf
  const float sl = scale * 1.4426950408889634f;
  s.scale_log2 = sl == 0.f ? 1.17549435e-38f : sl < 0.f ? -sl : sl;
  s.q_flip = sl < 0.f ? 0x80008000u : 0u;
  s.v_scale = v_scale, s.ldp = ldp, s.ldo = ldo;
  const dim3 grid((unsigned)(s.U - s.r + s.r * (ws ? s.most : 1)) * Hkv), block(wide::WAVES * WAVE);
  const auto* Q = static_cast<const __bf16*>(q);
  const auto* QG = static_cast<const __bf16*>(qg);
  auto* O = static_cast<__bf16*>(out);
  if (kv8)
    wide::attn_prefill_wide_kernel<true><<<grid, block, 0, stream>>>(Q, kc, vc, pos, QG, O, ws, s);
  else
    wide::attn_prefill_wide_kernel<false><<<grid, block, 0, stream>>>(Q, kc, vc, pos, QG, O, ws, s);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || !ws || !s.r) return e;
  wide::attn_prefill_wide_combine<<<dim3(s.r * wide::WAVES, Hkv, 16 / wide::CW), wide::CW * WAVE, 0,
                                    stream>>>(pos, QG, O, ws, s);
  return hipGetLastError();
}
