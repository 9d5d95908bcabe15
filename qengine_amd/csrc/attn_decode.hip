// Gated flash-decoding over a bf16 KV cache for n = 1..8 query rows on gfx950 (MI355X).
//
// Semantics follow the reference (csrc/attn.cu:1-9,58-149): row t sits at position pos+t and
// attends cache positions [0, min(pos+t+1, max_len)); scores are q.k * scale; the output is
// bf16(bf16(softmax . V) * bf16(sigmoid(gate))).
//
// Design (MI355X-first, not a translation of the reference's warp-per-position loop):
//  * One workgroup per (split-KV slice, KV head). Row t attends L_t positions, cut into slices of
//    split_size(L_t, NS) positions (the reference cuts ceil(L_t/NS), attn.cu:78-80; here that is
//    rounded up to whole 32-position tiles), so about NS slices hold work whatever the cache
//    capacity. A row's slices depend on its own length only: row t of an n-row call is
//    bit-identical to a 1-row call at position pos+t. The n <= 8 rows of a call use at most two
//    slice sizes; rows of one size share each K/V tile, and a call whose rows straddle a size
//    change runs one pass per size.
//  * The Hq/Hkv query heads of the GQA group times the n rows form the columns of the MFMA tiles
//    (NT tiles of 16 columns). K and V are read from HBM exactly once per call; Q stays in
//    registers as an MFMA operand.
//  * S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_16x16x32_bf16. With ~6 FLOP per byte, GQA-6
//    decode would otherwise need ~70% of the non-packed fp32 VALU peak at 8 TB/s.
//  * K is read with fully coalesced 16-byte non-temporal buffer loads (two 512-byte rows per
//    wave instruction) that write straight into a per-wave LDS tile (LDS DMA, no registers);
//    the lane-to-address assignment applies an XOR swizzle, so the MFMA operand is read from LDS
//    without bank conflicts. V is loaded straight into registers as 256-byte row
//    runs of 4 positions and regrouped by v_perm into position pairs for the MFMA A operand.
//  * Online softmax in the log2 domain per column. Row max/sum reductions over the 4 lane groups
//    use cross-lane shuffles. Rescaling of the accumulators is skipped when no column's max
//    moved (an exact no-op).
//  * Buffer resources bound the K/V reads to the slice: positions past it load as 0.
//  * A second launch merges the slices (log-sum-exp) and applies the sigmoid gate.
#include <algorithm>
#include <mutex>
#include <utility>

#include "attn_split.hpp"
#include "attn_tile.hpp"
#include "qe_attn.h"

namespace qe {

// Waves per workgroup. Tile k of a slice goes to wave k % 4 and the waves are merged in order
// 0..3 for every column-tile count NT: the within-slice decomposition (and so every rounding)
// is the same for 1 row and for 8, which is what keeps row t of an n-row call bit-identical to
// a 1-row call. (Eight waves for NT = 1 were measured no faster on MI355X.)
template <int NT>
constexpr int waves_for() { return 4; }
using tile::ROW_CHUNKS;


// One pass of a workgroup: rows [r0, r1) of the call share the slice size ch; this workgroup's
// slice s of them is [beg, end) (empty when beg >= end). Lmin is row r0's attended length.
struct Pass {
  int r0, r1, ch, beg, end, Lmin;
};

__device__ __forceinline__ Pass make_pass(int r0, int r1, int ch, int pos0, int max_len, int s) {
  Pass P;
  P.r0 = r0;
  P.r1 = r1;
  P.ch = ch;
  P.Lmin = min(pos0 + r0 + 1, max_len);
  const int Lhi = min(pos0 + r1, max_len);
  P.beg = s * ch;
  P.end = min(P.beg + ch, Lhi);
  return P;
}

// The call's passes: rows [0, tB) use slices of ch0 = split_size(L_0, NS) positions, rows [tB, n)
// slices of ch0 + 32. split_size(L) == ch0 exactly while L <= ch0 * NS, and n <= 8 consecutive
// lengths never reach a third size, so one division serves the whole call. Uniform.
__device__ __forceinline__ void call_split(int pos0, int n, int max_len, int NS, NsDiv nd,
                                           int& ch0, int& tB) {
  ch0 = split_size(min(pos0 + 1, max_len), nd);
  const long long lim = (long long)ch0 * NS;  // longest length with slices of ch0
  tB = n;
  if (max_len > lim && pos0 + n > lim) tB = (int)(lim - pos0);  // row tB is the first past lim
}

__device__ __forceinline__ Pass pass_of(int pi, int ch0, int tB, int n, int pos0, int max_len,
                                        int s) {
  return pi == 0 ? make_pass(0, tB, ch0, pos0, max_len, s)
                 : make_pass(tB, n, ch0 + TILE, pos0, max_len, s);
}

// Column col = t*grp + j (row t) belongs to the pass: its partial is stored.
__device__ __forceinline__ bool in_pass(int col, int grp, const Pass& P) {
  return col >= P.r0 * grp && col < P.r1 * grp;
}

// Slices that can hold work: a row attends at most max_len positions, in slices of >= 32.
static inline int max_slices(int max_len, int NS) {
  const int tiles = (max_len + TILE - 1) / TILE;
  return NS < tiles ? NS : tiles;
}

// Registers of one wave step (32 cache positions of one KV head). K goes straight to LDS.
struct VTile {
  u32x4_t v[8][2];  // V rows P(g4, e) = p0 + 16(e>>2) + 4g4 + (e&3), dims 128h + 8c + [0, 8)
};

// Buffer resource of one tile: based at row p0 of a head's cache (row_bytes per row), ending at
// row p_end, so loads at rows >= p_end read 0, exactly as a resource over the whole pass would.
// Every load's offset is then a loop-invariant lane term plus an immediate, and the per-tile
// address arithmetic is scalar (p0 is wave-uniform).
// A tile at or past p_end gets an empty resource: its loads read 0 and touch no memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const char* head_base, int p0,
                                                            int p_end, uint32_t row_bytes) {
  return make_rsrc_uniform(head_base + (size_t)p0 * row_bytes,
                           (uint32_t)max(p_end - p0, 0) * row_bytes);
}

// Lane terms of load_tile's offsets. K instruction j covers rows 2j, 2j+1 (lane i fetches the
// chunk that belongs in LDS slot 64j + i): row r = 2j + (i>>5), chunk (i&31) ^ (r&15), i.e. byte
// 1024j + (kl ^ 32(j&7)) with kl = 512(i>>5) + 16((i&31) ^ (i>>5)) (the swizzle moves bits 5-7
// only). V register e, h: row 16(e>>2) + 4g4 + (e&3), dims 128h + 8c: byte
// vl + 8192(e>>2) + 512(e&3) + 256h with vl = 2048g4 + 16c.
struct TileLanes {
  uint32_t kl, vl;
  __device__ __forceinline__ explicit TileLanes(int lane)
      : kl(512u * (lane >> 5) + 16u * ((lane & 31) ^ (lane >> 5))),
        vl(2048u * (lane >> 4) + 16u * (lane & 15)) {}
};

// Issue one tile's loads: 16 LDS-DMA loads of K (each reads 1 KB of contiguous cache into the
// wave's K tile at LDS byte ks_s), then 16 register loads of V (4 rows x 256 B per instruction).
// krs / vrs are the tile's resources (tile_rsrc). The scheduling barrier keeps every K load ahead
// of every V load: wait_and_compute's vmcnt wait counts on that order, which nothing else gives
// (the loads are independent, and the scheduler has interleaved them).
__device__ __forceinline__ void load_tile(VTile& b, uint32_t ks_s, __amdgpu_buffer_rsrc_t krs,
                                          __amdgpu_buffer_rsrc_t vrs, const TileLanes& tl) {
#pragma unroll
  for (int j = 0; j < 16; ++j)
    buffer_load16_to_lds_at(krs, (tl.kl ^ (32u * (j & 7))) + 1024u * j, ks_s + 1024u * j);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      b.v[e][h] = buffer_load16_stream(vrs, tl.vl + 8192u * (e >> 2) + 512u * (e & 3) + 256u * h);
}

// The two halves of load_tile for the look-ahead loop (run_pass): K of a tile into one of the
// wave's two LDS K slots, and V of a tile into registers.
// The lane terms pass through an empty asm so that they are formed at each issue: otherwise the
// compiler hoists all 16 + 16 offsets out of the tile loop and keeps them live (28 more registers).
__device__ __forceinline__ void issue_k(uint32_t ks_s, __amdgpu_buffer_rsrc_t krs,
                                        const TileLanes& tl) {
  uint32_t kl = tl.kl;
  asm volatile("" : "+v"(kl));
#pragma unroll
  for (int j = 0; j < 16; ++j)
    buffer_load16_to_lds_at(krs, (kl ^ (32u * (j & 7))) + 1024u * j, ks_s + 1024u * j);
}
__device__ __forceinline__ void issue_v(VTile& b, __amdgpu_buffer_rsrc_t vrs, const TileLanes& tl) {
  uint32_t vl = tl.vl;
  asm volatile("" : "+v"(vl));  // two bases (vl, vl + 8192) and immediate offsets
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      b.v[e][h] = buffer_load16_stream(vrs, vl + 8192u * (e >> 2) + 512u * (e & 3) + 256u * h);
}

// Order this wave's LDS accesses: the compiler must not move LDS reads/writes across it (lanes
// exchange data through LDS, which single-thread alias analysis cannot see).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Compute one tile whose K has landed in the wave's LDS slot ks_lds and whose V registers are
// loaded (the compiler waits for those). Masking is needed only on tiles reaching past the
// shortest attended length among the real columns (Lmin).
template <int NT>
__device__ __forceinline__ void compute_tile(const VTile& b, const u32x4_t* ks_lds, int p0,
                                             int Lmin, const int (&Lcol)[NT],
                                             const bf16x8_t (&qb)[NT][8], float scale_log2,
                                             int c, int g4, float (&m)[NT], float (&l)[NT],
                                             f32x4_t (&acc)[NT][16]) {
  wave_lds_fence();
  f32x4_t sacc[NT][2];
  // (K tiles 256-byte aligned.) Two column tiles: the K reads are scheduled two ahead of their
  // MFMA pairs (tile::qk_tile LEAD). Same-box harness A/B, partials us, none -> 2: 3 rows at
  // 16387 17.73 -> 17.45, 5 rows at 16389 18.28 -> 18.01, 4 rows at 8196 13.41 -> 13.25, 5 rows
  // at 32773 27.64 -> 27.44 (leads 4 and 6: no gain); bits identical. One tile: no change.
  tile::qk_tile<NT, NT == 1, NT == 2 ? 2 : 0>(ks_lds, qb, c, g4, sacc);
  wave_lds_fence();  // this tile's K reads happen before the next tile's LDS-DMA writes
  u32x4_t pb_hi[NT], pb_lo[NT];
  if (p0 + TILE > Lmin)
    tile::softmax_tile<NT, true, true>(sacc, p0, Lcol, scale_log2, g4, m, l, acc, pb_hi, pb_lo);
  else
    tile::softmax_tile<NT, false, true>(sacc, p0, Lcol, scale_log2, g4, m, l, acc, pb_hi, pb_lo);
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    u32x4_t vr[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) vr[e] = b.v[e][hh];
    tile::pv_half<NT, true>(vr, hh, pb_hi, pb_lo, acc);
  }
}

// Wait for the tile's K (its 16 LDS-DMA loads were issued before the 16 V loads, so at most 16
// loads may remain in flight), then compute the tile.
template <int NT>
__device__ __forceinline__ void wait_and_compute(const VTile& b, const u32x4_t* ks_lds, int p0,
                                                 int Lmin, const int (&Lcol)[NT],
                                                 const bf16x8_t (&qb)[NT][8], float scale_log2,
                                                 int c, int g4, float (&m)[NT], float (&l)[NT],
                                                 f32x4_t (&acc)[NT][16]) {
  vmcnt_wait<16>();
  compute_tile<NT>(b, ks_lds, p0, Lmin, Lcol, qb, scale_log2, c, g4, m, l, acc);
}

// Fused prep + decode: the wave's first tile is loaded before the prep. Its K goes to registers
// (KRegs: chunk k[j] of lane i is the one load_tile's LDS-DMA instruction j would put in slot
// 64j + i), not to LDS by DMA: the compiler cannot tell the DMA's LDS target from the prep's LDS
// and would make the prep's first LDS read wait for the tile.
struct KRegs {
  u32x4_t k[16];
};
__device__ __forceinline__ void load_tile_regs(KRegs& kr, VTile& b, __amdgpu_buffer_rsrc_t krs,
                                               __amdgpu_buffer_rsrc_t vrs, int p0, int lane, int c,
                                               int g4) {
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int r = 2 * j + (lane >> 5);
    const int q = (lane & 31) ^ (r & 15);
    kr.k[j] = buffer_load16_stream(krs, (uint32_t)(p0 + r) * (HD * 2) + q * 16);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      b.v[e][h] = buffer_load16_stream(
          vrs, (uint32_t)(p0 + 16 * (e >> 2) + 4 * g4 + (e & 3)) * (HD * 2) + (128 * h + 8 * c) * 2);
}

// After the prep: the tile's rows at the positions the prep wrote (pos0 + t, t in [t_lo, t_hi))
// hold stale bytes; their K rows (staged by the prep, FusedLds::knew) and V rows (vnew) replace
// them in the registers, so the tile holds what a load after the write would have read. Positions
// at or past the pass's end (p_end) keep the zeros the bounded load returned, as in the unfused
// decode. K then goes to the wave's LDS tile.
__device__ __forceinline__ void fused_place_tile(KRegs& kr, VTile& b, u32x4_t* ks_lds,
                                                 const u32x4_t (*knew)[ROW_CHUNKS],
                                                 const u32x4_t (*vnew)[ROW_CHUNKS], int p0,
                                                 int p_end, int pos0, int t_lo, int t_hi,
                                                 int lane, int c, int g4) {
  t_hi = min(t_hi, p_end - pos0);
  if (t_hi > t_lo) {  // uniform
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int r = 2 * j + (lane >> 5);
      const int t = p0 + r - pos0;
      if (t >= t_lo && t < t_hi) kr.k[j] = knew[t][(lane & 31) ^ (r & 15)];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int t = p0 + 16 * (e >> 2) + 4 * g4 + (e & 3) - pos0;
      if (t >= t_lo && t < t_hi) {
#pragma unroll
        for (int h = 0; h < 2; ++h) b.v[e][h] = vnew[t][16 * h + c];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 16; ++j) ks_lds[64 * j + lane] = kr.k[j];
}

// fp8 KV (E4M3FN codes, 256-byte rows): the same tile and the same arithmetic after an exact
// conversion to bf16. K: 8 LDS-DMA loads (instruction j covers rows 4j..4j+3; lane i fetches the
// 16-byte chunk that belongs in slot 64j + i, chunks XOR-swizzled by row as for bf16); V: 16
// register loads of 8 bytes, the dims and rows of the bf16 layout (VTile), converted before use.
struct VTile8 {
  u32x2_t v[8][2];  // V rows P(g4, e), dims 128h + 8c + [0, 8), as fp8 codes
};

// Lane terms of the fp8 tile loads' offsets (tile resources as for bf16). K instruction j: row
// r = 4j + (i>>4), chunk (i&15) ^ (r&15), i.e. byte 1024j + (kl ^ 64(j&3)) with
// kl = 256(i>>4) + 16((i&15) ^ (i>>4)). V register e, h: byte vl + 4096(e>>2) + 256(e&3) + 128h
// with vl = 1024g4 + 8c.
struct TileLanes8 {
  uint32_t kl, vl;
  __device__ __forceinline__ explicit TileLanes8(int lane)
      : kl(256u * (lane >> 4) + 16u * ((lane & 15) ^ (lane >> 4))),
        vl(1024u * (lane >> 4) + 8u * (lane & 15)) {}
};

// S^T = K Q^T from an fp8 K tile in LDS: lane (c, g4) reads the 8 codes of row 16T + c, dims
// [32ks + 8g4, +8) (half of the swizzled 16-byte chunk 2ks + g4/2) and converts them to the bf16
// A operand of qk_tile. With the tile 256-byte aligned, chunk (2ks + g4/2) ^ c at byte 16 chunk
// is one per-lane base XORed with 32 ks (the swizzle moves bits 5-7 only) plus 4096 T.
template <int NT>
__device__ __forceinline__ void qk_tile8(const u32x4_t* k_lds, const bf16x8_t (&qb)[NT][8], int c,
                                         int g4, f32x4_t (&sacc)[NT][2]) {
  typedef __attribute__((address_space(3))) const u32x2_t lds_u32x2;
  const uint32_t b0 =
      (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const char*)reinterpret_cast<const char*>(k_lds)) +
      c * 256 + 16 * (c & 14) + 16 * ((g4 >> 1) ^ (c & 1)) + 8 * (g4 & 1);
#pragma unroll
  for (int T = 0; T < 2; ++T) {
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) sacc[ct][T] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const u32x2_t w = *(lds_u32x2*)(uintptr_t)((b0 ^ (32u * ks)) + 4096 * T);
      const bf16x8_t kop = as_bf16x8(fp8x8_to_bf16x8(w));
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) sacc[ct][T] = mfma16x16x32(kop, qb[ct][ks], sacc[ct][T]);
    }
  }
}

// One fp8 tile's loads for the look-ahead loop: the K codes (8 KB) into one of the wave's two LDS
// K slots (8 LDS-DMA loads), and the V codes into registers (16 loads of 8 bytes).
__device__ __forceinline__ void issue_k8(uint32_t ks_s, __amdgpu_buffer_rsrc_t krs,
                                         const TileLanes8& tl) {
  uint32_t kl = tl.kl;
  asm volatile("" : "+v"(kl));
#pragma unroll
  for (int j = 0; j < 8; ++j)
    buffer_load16_to_lds_at(krs, (kl ^ (64u * (j & 3))) + 1024u * j, ks_s + 1024u * j);
}
__device__ __forceinline__ void issue_v8(VTile8& b, __amdgpu_buffer_rsrc_t vrs,
                                         const TileLanes8& tl) {
  uint32_t vl = tl.vl;
  asm volatile("" : "+v"(vl));
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      b.v[e][h] = buffer_load8_stream(vrs, vl + 4096u * (e >> 2) + 256u * (e & 3) + 128u * h);
}

// One fp8 tile whose K codes have landed in the wave's LDS slot ks_lds (as compute_tile).
template <int NT>
__device__ __forceinline__ void compute_tile8(const VTile8& b, const u32x4_t* ks_lds, int p0,
                                              int Lmin, const int (&Lcol)[NT],
                                              const bf16x8_t (&qb)[NT][8], float scale_log2,
                                              int c, int g4, float (&m)[NT], float (&l)[NT],
                                              f32x4_t (&acc)[NT][16]) {
  wave_lds_fence();
  f32x4_t sacc[NT][2];
  qk_tile8<NT>(ks_lds, qb, c, g4, sacc);
  wave_lds_fence();  // this tile's K reads happen before the next tile's LDS-DMA writes
  u32x4_t pb_hi[NT], pb_lo[NT];
  if (p0 + TILE > Lmin)
    tile::softmax_tile<NT, true, true>(sacc, p0, Lcol, scale_log2, g4, m, l, acc, pb_hi, pb_lo);
  else
    tile::softmax_tile<NT, false, true>(sacc, p0, Lcol, scale_log2, g4, m, l, acc, pb_hi, pb_lo);
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    u32x4_t vr[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) vr[e] = fp8x8_to_bf16x8(b.v[e][hh]);
    tile::pv_half<NT, true>(vr, hh, pb_hi, pb_lo, acc);
  }
}

// LDS: per-wave K tiles during the loop; reused for the cross-wave merge afterwards. The tile
// loop keeps the next tile's K in flight in a second slot (two 16 KB bf16 slots, or two 8 KB fp8
// slots, per wave); the fused prep + decode keeps one bf16 slot (its prep needs the rest).
constexpr int lds_wave_bytes(bool fused, bool kv8) {
  return kv8 ? 2 * TILE * HD : (fused ? 1 : 2) * TILE * HD * 2;
}
template <int WAVES>
constexpr int lds_k_bytes() { return WAVES * TILE * HD * 2; }  // 16 KB per wave

// Inputs of the prep fused into the partials kernel (qe_attn_prep_decode); unused otherwise.
struct PrepIn {
  const __bf16* qg;   // rows [n][ldp]: per q head [q (256) | gate (256)]
  const __bf16* k;    // rows [n][ldp]: Hkv*256
  const __bf16* v;
  long ldp;
  const __bf16* qnw;
  const __bf16* knw;
  const float* inv_freq;
  __bf16* q_out;      // [n][Hq*256]
  int rd;
  float eps;
};

// LDS of the fused prep: the group's q rows (bf16, 16-byte chunks, rows padded by one chunk so the
// 16 columns a lane group reads hit different banks), per wave: the two norm weight rows and
// inv_freq, one 256-float row per half-wave for the rotate-half exchange; and the rotary cos/sin
// table of the call's rows.
constexpr int FQ_ROW_U4 = ROW_CHUNKS + 1;
constexpr int PREP_WAVES = 4;
constexpr int ROPE_TAB = 256;  // n * rd/2 entries, one per thread (the fused path's limit)
constexpr int FUSED_NEW_ROWS = 8;  // rows of a call (n <= 8)
template <int NT>
struct PrepShape {
  static constexpr int MAXI = (16 * NT + 8 + PREP_WAVES - 1) / PREP_WAVES;  // items per wave
  static constexpr int PAIRS = (MAXI + 1) / 2;  // 16-byte loads of two rows per lane
};
template <int NT>
struct FusedLds {
  u32x4_t q[16 * NT][FQ_ROW_U4];
  u32x4_t stage_w[PREP_WAVES][2][ROW_CHUNKS];  // qnw, knw
  float stage_f[PREP_WAVES][HD / 2];          // inv_freq (half <= 128)
  float xn[PREP_WAVES][2][HD];  // per half-wave item: the normalised row (rotate_half partner)
  float cs[ROPE_TAB], sn[ROPE_TAB];
  u32x4_t knew[FUSED_NEW_ROWS][ROW_CHUNKS];  // the cache rows this workgroup writes, by row t:
  u32x4_t vnew[FUSED_NEW_ROWS][ROW_CHUNKS];  // patched into the tile loaded before the prep
};
__shared__ __attribute__((aligned(16))) char fused_lds_raw[sizeof(FusedLds<1>)];
template <int NT>
__device__ __forceinline__ FusedLds<NT>& fused_lds() {
  return *reinterpret_cast<FusedLds<NT>*>(fused_lds_raw);
}
__device__ __forceinline__ u32x4_t fused_q_lds(int col, int chunk) {
  return reinterpret_cast<const u32x4_t*>(fused_lds_raw)[col * FQ_ROW_U4 + chunk];
}

// The prep of qe_attn_prep for this workgroup, one row ("item") per half-wave at a time and no
// workgroup barrier inside an item: items are the ncols q rows of KV head g's group (to LDS, and
// to q_out from slice 0) and the cache rows pos+t, t in [t_lo, t_hi), that lie in this slice;
// items 2P*4 + w and (2P+1)*4 + w go to the two halves of wave w (fused_prep_pair).
// The input rows are loaded with 16-byte loads (lanes 0-31 one row, 32-63 the next; lane 32h + L
// holds dims 8L .. 8L+7 of its row, the layout the items compute in), after the norm weights and
// inv_freq (loads return in order: the rotary table waits only for those) and before the caller's
// tile prefetch (a later load would wait for the tile, and a wave can have only 63 loads
// outstanding). The V rows are loaded at the end, only by the workgroup that writes cache rows.
template <int NT>
struct PrepRegs {
  u32x4_t x[PrepShape<NT>::PAIRS], w, f;
};

template <int NT>
__device__ __forceinline__ void fused_prep_load(PrepRegs<NT>& r, const PrepIn& pin, int g,
                                                int grp, int n, int ncols, int t_lo, int t_hi) {
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const int nitems = ncols + (t_hi - t_lo);
  const int hl = lane >> 5, ch = lane & 31;  // row of the pair, 16-byte chunk of the row
  r.w = reinterpret_cast<const u32x4_t*>(hl ? pin.knw : pin.qnw)[ch];
  const int half = pin.rd >> 1;  // a multiple of 4 on this path
  // lanes past the table load (and stage) its last chunk again, so the staging store needs no
  // branch that the compiler could sink this load into
  r.f = reinterpret_cast<const u32x4_t*>(pin.inv_freq)[min(lane, half / 4 - 1)];
#pragma unroll
  for (int P = 0; P < PrepShape<NT>::PAIRS; ++P) {
    int it = (2 * P + hl) * PREP_WAVES + w;
    it = it < nitems ? it : 0;  // slots past the end load row 0's q (discarded)
    const bool isq = it < ncols;
    const int t = isq ? it / grp : t_lo + (it - ncols);
    const __bf16* src = isq ? pin.qg + (size_t)t * pin.ldp + (size_t)(g * grp + it % grp) * 2 * HD
                            : pin.k + (size_t)t * pin.ldp + (size_t)g * HD;
    r.x[P] = reinterpret_cast<const u32x4_t*>(src)[ch];
  }
}

// One pair of items per wave, one item per half-wave: half hl of wave w takes item
// (2P + hl) * PREP_WAVES + w, whose input row its lanes loaded themselves (fused_prep_load: lane
// (hl, ch) holds dims 8ch .. 8ch+7), so the row needs no staging. The sum of squares follows the
// prep kernel's reduction exactly (attn_prep_rows_kernel: dims c^32, c^16, c^8 in lanes ^4, ^2,
// ^1, then c^4, c^2, c^1 within the lane, and ((r0 + r1) + r2) + r3 over the four 64-dim groups),
// so every output is bit-identical to qe_attn_prep. 16-byte LDS and global stores.
template <int NT, int P>
__device__ __forceinline__ void fused_prep_pair(const PrepRegs<NT>& r, const PrepIn& pin, int s,
                                                int g, int grp, int Hq, int ncols, int nitems,
                                                int pos0, int t_lo, int max_len, __bf16* kc,
                                                __bf16* vc) {
  FusedLds<NT>& L = fused_lds<NT>();
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const int hl = lane >> 5, ch = lane & 31;
  const int it = (2 * P + hl) * PREP_WAVES + w;
  if (it >= nitems) return;  // uniform per half-wave
  const int rd = pin.rd, half = rd >> 1;
  float* xn = L.xn[w][hl];
  const bool isq = it < ncols;
  const int t = isq ? it / grp : t_lo + (it - ncols);
  const u32x4_t wr = L.stage_w[w][isq ? 0 : 1][ch];
  float x[8], wg[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[2 * i] = lo_bf16(r.x[P][i]);
    x[2 * i + 1] = hi_bf16(r.x[P][i]);
    wg[2 * i] = lo_bf16(wr[i]);
    wg[2 * i + 1] = hi_bf16(wr[i]);
  }
  float sq[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) sq[q] = x[q] * x[q];
#pragma unroll
  for (int q = 0; q < 8; ++q) sq[q] = sq[q] + dpp<0x1B>(dpp<0x141>(sq[q]));  // lane ^ 4: dim ^ 32
#pragma unroll
  for (int q = 0; q < 8; ++q) sq[q] = sq[q] + dpp<0x4E>(sq[q]);              // lane ^ 2: dim ^ 16
#pragma unroll
  for (int q = 0; q < 8; ++q) sq[q] = sq[q] + dpp<0xB1>(sq[q]);              // lane ^ 1: dim ^ 8
  float u[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) u[q] = sq[q] + sq[q + 4];                      // dim ^ 4
  const float gsum = (u[0] + u[2]) + (u[1] + u[3]);                          // dim ^ 2, then ^ 1
  const int base = lane & 32;
  const float r0 = __shfl(gsum, base), r1 = __shfl(gsum, base + 8);
  const float r2 = __shfl(gsum, base + 16), r3 = __shfl(gsum, base + 24);
  const float total = ((r0 + r1) + r2) + r3;
  const float inv = 1.0f / sqrtf(total / (float)HD + pin.eps);
  float xv[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) xv[q] = round_bf16((x[q] * inv) * (1.0f + wg[q]));
  // the half-wave's LDS row: the previous pair's partner reads are done before it is rewritten
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  *reinterpret_cast<f32x4_t*>(&xn[8 * ch]) = f32x4_t{xv[0], xv[1], xv[2], xv[3]};
  *reinterpret_cast<f32x4_t*>(&xn[8 * ch + 4]) = f32x4_t{xv[4], xv[5], xv[6], xv[7]};
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  float y[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) y[q] = xv[q];
  const int d0 = 8 * ch;
  if (d0 < rd) {
    if ((half & 7) == 0) {  // the lane's 8 dims lie on one side of half: 16-byte LDS reads
      const bool lo = d0 < half;
      const int e0 = t * half + (lo ? d0 : d0 - half);
      const float* pp = &xn[lo ? d0 + half : d0 - half];
      const f32x4_t p[2] = {*reinterpret_cast<const f32x4_t*>(pp),
                            *reinterpret_cast<const f32x4_t*>(pp + 4)};
      const f32x4_t c[2] = {*reinterpret_cast<const f32x4_t*>(&L.cs[e0]),
                            *reinterpret_cast<const f32x4_t*>(&L.cs[e0 + 4])};
      const f32x4_t sn[2] = {*reinterpret_cast<const f32x4_t*>(&L.sn[e0]),
                             *reinterpret_cast<const f32x4_t*>(&L.sn[e0 + 4])};
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const float rot = lo ? -p[q >> 2][q & 3] : p[q >> 2][q & 3];  // rotate_half
        y[q] = round_bf16(round_bf16(xv[q] * c[q >> 2][q & 3]) + round_bf16(rot * sn[q >> 2][q & 3]));
      }
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int d = d0 + q;
        if (d < rd) {
          const int e = t * half + (d < half ? d : d - half);
          const float rot = d < half ? -xn[d + half] : xn[d - half];  // rotate_half
          y[q] = round_bf16(round_bf16(xv[q] * L.cs[e]) + round_bf16(rot * L.sn[e]));
        }
      }
    }
  }
  u32x4_t yo;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    yo[i] = (uint32_t)__builtin_bit_cast(uint16_t, f32_to_bf16(y[2 * i])) |
            ((uint32_t)__builtin_bit_cast(uint16_t, f32_to_bf16(y[2 * i + 1])) << 16);
  if (isq) {
    const int head = g * grp + it % grp;
    L.q[it][ch] = yo;
    if (s == 0)
      *reinterpret_cast<u32x4_t*>(pin.q_out + (size_t)t * Hq * HD + (size_t)head * HD + 8 * ch) = yo;
  } else {
    const size_t dst = ((size_t)g * max_len + (pos0 + t)) * HD + 8 * ch;
    const u32x4_t vb = *reinterpret_cast<const u32x4_t*>(
        pin.v + (size_t)t * pin.ldp + (size_t)g * HD + 8 * ch);  // v bit for bit
    *reinterpret_cast<u32x4_t*>(kc + dst) = yo;
    *reinterpret_cast<u32x4_t*>(vc + dst) = vb;
    L.knew[t][ch] = yo;
    L.vnew[t][ch] = vb;
  }
}

// The norm weights and inv_freq into this wave's LDS staging area (waits for those two loads).
template <int NT>
__device__ __forceinline__ void fused_prep_stage(const PrepRegs<NT>& r, const PrepIn& pin) {
  FusedLds<NT>& L = fused_lds<NT>();
  const int lane = threadIdx.x & (WAVE - 1), w = threadIdx.x / WAVE;
  const int hl = lane >> 5, ch = lane & 31, half = pin.rd >> 1;
  L.stage_w[w][hl][ch] = r.w;
  reinterpret_cast<u32x4_t*>(L.stage_f[w])[min(lane, half / 4 - 1)] = r.f;  // same bits per slot
}

// After fused_prep_stage: the rotary cos/sin table of the call's rows, then a workgroup barrier.
template <int NT>
__device__ __forceinline__ void fused_prep_table(const PrepIn& pin, int n, int pos0) {
  FusedLds<NT>& L = fused_lds<NT>();
  const int w = threadIdx.x / WAVE;
  const int half = pin.rd >> 1;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int e = threadIdx.x;  // rotary table entry (row e / half, frequency e % half)
  if (e < n * half) {
    const RopeCS cs = rope_cs_f(pos0 + e / half, L.stage_f[w][e % half], pin.rd, 0);
    L.cs[e] = cs.cs;
    L.sn[e] = cs.sn;
  }
  lds_barrier();
}

// After fused_prep_table. Ends with a workgroup barrier after which the q rows are readable in
// LDS and, in the workgroup that writes cache rows, those writes have completed (so the waves'
// later tile loads see them).
template <int NT, int... Ps>
__device__ __forceinline__ void fused_prep_compute(const PrepRegs<NT>& r, const PrepIn& pin, int s,
                                                   int g, int grp, int n, int Hq, int ncols,
                                                   int pos0, int t_lo, int t_hi, int max_len,
                                                   __bf16* kc, __bf16* vc,
                                                   std::integer_sequence<int, Ps...>) {
  const int nitems = ncols + (t_hi - t_lo);
  (fused_prep_pair<NT, Ps>(r, pin, s, g, grp, Hq, ncols, nitems, pos0, t_lo, max_len, kc, vc),
   ...);
  if (t_hi > t_lo)
    __syncthreads();  // release: the cache rows are written before any wave loads them
  else
    lds_barrier();    // only the q rows in LDS are shared; tile loads stay in flight
}

// part_o [n][Hq][NS][HD] (unnormalised O), part_ml [n][Hq][NS][2] = (max in log2 units, sum).
// NT = 1 (decode, 1-2 rows at GQA 6) fits in 256 registers, which lets two workgroups share a CU;
// NT = 2 (3-5 rows) needs the whole register file. Wider shapes use attn_partials_cols_kernel.
// Columns of rows outside the current pass are computed along (columns never mix) and not stored.
//
// FUSED: the kernel also does qe_attn_prep's work (the q rows in registers come from qg through
// the same RMSNorm1p + RoPE code, the new K/V rows are written to the cache), so prep + decode is
// two launches. Each workgroup computes the q rows of its GQA group (slice 0 also writes q_out).
// Every workgroup whose slices hold a position pos+t writes cache row pos+t itself, before any of
// its waves loads a tile, so it never depends on another workgroup's write (when two workgroups
// write one row, they write the same bits). kc/vc are written here, so they are not __restrict__.
template <int NT, bool FUSED = false, bool MULTI = true, bool KV8 = false,
          int WAVES = waves_for<NT>()>
__global__ void __launch_bounds__(WAVES * WAVE) __attribute__((amdgpu_waves_per_eu(NT == 1 && KV8 ? 2 : 1, 2)))
attn_partials_kernel(const __bf16* __restrict__ q, const __bf16* kc, const __bf16* vc,
                     const int* __restrict__ pos_ptr, float* __restrict__ part_o,
                     float* __restrict__ part_ml, int n, int Hq, int Hkv, int max_len, int NS,
                     NsDiv nd, float scale_log2, PrepIn pin, int row0) {
  const int pos0 = pos_ptr[0] + row0;  // first: the slicing waits for it
  const int s = blockIdx.x, g = blockIdx.y;
  const int grp = Hq / Hkv;
  // The wave index as a wave-uniform value, so that tile positions and the addresses derived
  // from them stay in scalar registers and the tile loop is a scalar loop.
  const int lane = threadIdx.x & (WAVE - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int c = lane & 15, g4 = lane >> 4;
  const int ncols = grp * n;

  // Q^T as the MFMA B operand. Column ct*16+c is (row t, head g*grp+j), col = t*grp + j.
  // Lane group g4 holds dims [32ks + 8g4, +8) of k-step ks (the same dims as the K operand).
  // Loaded before pos arrives (it does not depend on it); the fused kernel preps it further down.
  bf16x8_t qb[NT][8];
  int trow[NT];  // the column's row (n for padding columns)
#pragma unroll
  for (int ct = 0; ct < NT; ++ct) {
    const int col = ct * 16 + c;
    const int t = col / grp, j = col - t * grp;
    trow[ct] = col < ncols ? t : n;
    if (!FUSED && col < ncols) {
      const u32x4_t* src =
          reinterpret_cast<const u32x4_t*>(q + (size_t)t * Hq * HD + (size_t)(g * grp + j) * HD);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) qb[ct][ks] = as_bf16x8(src[4 * ks + g4]);
    } else {
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) qb[ct][ks] = as_bf16x8(u32x4_t{0u, 0u, 0u, 0u});
    }
  }

  int ch0, tB;
  call_split(pos0, n, max_len, NS, nd, ch0, tB);
  if constexpr (!MULTI) tB = 1;  // one row: one pass
  const int npass = tB < n ? 2 : 1;
  const Pass PA = pass_of(0, ch0, tB, n, pos0, max_len, s);
  const Pass PB = pass_of(1, ch0, tB, n, pos0, max_len, s);
  const bool attendA = PA.beg < PA.end, attendB = MULTI && npass > 1 && PB.beg < PB.end;
  const bool attend = attendA || attendB;  // uniform per workgroup
  if (!attend && !(FUSED && s == 0)) return;  // (slice 0 of the fused kernel still writes q_out)

  constexpr int WAREA = lds_wave_bytes(FUSED, KV8);  // this wave's K slots
  static_assert(WAREA >= lds_k_bytes<1>(), "each wave's area holds its merge buffer (16 KB)");
  __shared__ __attribute__((aligned(256))) char lds[WAVES * WAREA];
  __shared__ float s_m[WAVES][16 * NT], s_l[WAVES][16 * NT];
  static_assert(!(FUSED && KV8), "the fused prep writes a bf16 cache");
  static_assert(!FUSED || NT == 1, "the fused prep runs at one column tile");
  u32x4_t* ks_lds = reinterpret_cast<u32x4_t*>(lds + w * WAREA);
  constexpr int ELEM = KV8 ? 1 : 2;  // bytes per cache value
  const size_t head_off = (size_t)g * max_len * HD * ELEM;  // bytes
  const char* kbase = reinterpret_cast<const char*>(kc) + head_off;  // this KV head's K rows
  const char* vbase = reinterpret_cast<const char*>(vc) + head_off;
  const uint32_t ks_s = lds_byte_uniform(ks_lds);  // the wave's K tile in LDS

  // K/V buffer resources of a pass: loads past the pass's last position read 0
  auto pass_rsrc = [&](const Pass P, const __bf16* base) __attribute__((always_inline)) {
    const uint32_t bytes = (uint32_t)P.end * (uint32_t)(HD * ELEM);
    return make_rsrc_uniform(reinterpret_cast<const char*>(base) + head_off, bytes);
  };
  VTile buf;        // V registers of the wave's current tile
  KRegs kpf;        // fused: K of the tile loaded before the prep
  bool pf = false;  // fused: the first tile of the first pass was loaded before the prep
  int t_lo = 0, t_hi = 0;
  if constexpr (FUSED) {
    // rows t in [t_lo, t_hi) sit at positions this workgroup reads: their K/V rows are written here
    const int lo = attendA ? PA.beg : PB.beg, hi = attendB ? PB.end : PA.end;
    t_lo = max(lo - pos0, 0);
    t_hi = attend ? max(min(hi - pos0, n), t_lo) : t_lo;  // empty when none is here
    PrepRegs<NT> pr;
    fused_prep_load<NT>(pr, pin, g, grp, n, ncols, t_lo, t_hi);
    fused_prep_stage<NT>(pr, pin);
    fused_prep_table<NT>(pin, n, pos0);
    // The wave's first tile does not depend on the prep (rows the prep writes are patched in
    // after it, fused_place_tile): its loads go out once the rotary table, which one wave
    // computes for all, is done and the input rows have arrived (so no wait for those rows can
    // also wait for the tile), and land while the items run.
    const Pass P0 = attendA ? PA : PB;
    const int pf_p0 = P0.beg + w * TILE;
    pf = attend && pf_p0 < P0.end;
    __builtin_amdgcn_sched_barrier(0);
    // The input rows arrived during the table; waiting for them here, before the conditional
    // tile loads, keeps the compiler from waiting for the tile too where the items read them.
#pragma unroll
    for (int P = 0; P < PrepShape<NT>::PAIRS; ++P) asm volatile("" ::"v"(pr.x[P]));
    if (pf) load_tile_regs(kpf, buf, pass_rsrc(P0, kc), pass_rsrc(P0, vc), pf_p0, lane, c, g4);
    __builtin_amdgcn_sched_barrier(0);
    fused_prep_compute<NT>(pr, pin, s, g, grp, n, Hq, ncols, pos0, t_lo, t_hi, max_len,
                           const_cast<__bf16*>(kc), const_cast<__bf16*>(vc),
                           std::make_integer_sequence<int, PrepShape<NT>::PAIRS>{});
    if (!attend) return;  // slice 0 beyond every attended position: q_out written, nothing else
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
      const int col = ct * 16 + c;
      if (col < ncols) {
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) qb[ct][ks] = as_bf16x8(fused_q_lds(col, 4 * ks + g4));
      }
    }
  }

  // One pass, inlined once per call of the lambda (as a loop over passes, the merge's
  // loop-invariant addresses would be hoisted and stay live through the tile loop).
  auto run_pass = [&](const Pass P, bool first) __attribute__((always_inline)) {
    int Lcol[NT];  // attended length of the pass's columns; 0 (all masked) for the others
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
      Lcol[ct] = in_pass(ct * 16 + c, grp, P) ? min(pos0 + trow[ct] + 1, max_len) : 0;

    float m[NT], l[NT];
    f32x4_t acc[NT][16];  // [8hh + i]: O^T dims 128hh + 32g4 + 8ii + i (tile::pv_half)
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
      m[ct] = -INFINITY;
      l[ct] = 0.f;
#pragma unroll
      for (int a = 0; a < 16; ++a) acc[ct][a] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    // Look-ahead tile loop (every partials kernel but the fused one). A wave's tiles are p0,
    // p0 + STEP, ...; K runs one tile ahead in the second of the wave's two LDS slots: as soon as
    // tile k's K has landed, tile k+1's K is issued, and tile k+1's V right after tile k's
    // O^T += V^T P^T has consumed the V registers. Issue order K0, V0 | K1 | V1 | K2 | ...: at the
    // top of each tile only that tile's V (16 loads) can have been issued after its K. Tile
    // k+1's K lands during tile k's arithmetic, and the last data a wave waits for is a V tile,
    // whose flight S^T and the softmax of its tile overlap. The last tile is peeled, so no load
    // is issued past the pass (a load with an empty resource still costs issue and return
    // slots: always issuing the next K cost 0.3-0.5 us per call). Same arithmetic as the
    // single-slot loop, bit for bit.
    constexpr int STEP = WAVES * TILE;
    auto lds_tile = [&](uint32_t b) __attribute__((always_inline)) {
      return (const u32x4_t*)((__attribute__((address_space(3))) const u32x4_t*)(uintptr_t)b);
    };
    if constexpr (KV8) {
      VTile8 buf;
      const TileLanes8 tl(lane);
      int p0 = P.beg + w * TILE;
      if (p0 < P.end) {
        uint32_t cur = ks_s, nxt = ks_s + TILE * HD;  // two 8 KB slots
        issue_k8(cur, tile_rsrc(kbase, p0, P.end, HD), tl);
        __builtin_amdgcn_sched_barrier(0);
        issue_v8(buf, tile_rsrc(vbase, p0, P.end, HD), tl);
        for (; p0 + STEP < P.end; p0 += STEP) {
          vmcnt_wait<16>();  // this tile's K: its V (16 loads) may remain
          __builtin_amdgcn_sched_barrier(0);
          issue_k8(nxt, tile_rsrc(kbase, p0 + STEP, P.end, HD), tl);
          __builtin_amdgcn_sched_barrier(0);
          compute_tile8<NT>(buf, lds_tile(cur), p0, P.Lmin, Lcol, qb, scale_log2, c, g4, m, l,
                            acc);
          __builtin_amdgcn_sched_barrier(0);
          issue_v8(buf, tile_rsrc(vbase, p0 + STEP, P.end, HD), tl);
          const uint32_t t = cur;
          cur = nxt;
          nxt = t;
        }
        vmcnt_wait<16>();
        compute_tile8<NT>(buf, lds_tile(cur), p0, P.Lmin, Lcol, qb, scale_log2, c, g4, m, l, acc);
      }
    } else if constexpr (FUSED) {
      // single slot: the fused prep's LDS leaves room for one K tile per wave
      int p0 = P.beg + w * TILE;
      if (first && pf) {  // the tile loaded before the prep
        fused_place_tile(kpf, buf, ks_lds, fused_lds<NT>().knew, fused_lds<NT>().vnew, p0, P.end,
                         pos0, t_lo, t_hi, lane, c, g4);
        wait_and_compute<NT>(buf, ks_lds, p0, P.Lmin, Lcol, qb, scale_log2, c, g4, m, l, acc);
        p0 += STEP;
      }
      // Where no tile was loaded before the prep, the compiler, which cannot tie this branch to
      // the prefetch's, counts those loads as pending: uses of the registers here take its wait
      // before the loop, not among the tile loop's K loads (no wait at run time on either path).
#pragma unroll
      for (int j = 0; j < 16; ++j) asm volatile("" ::"v"(kpf.k[j]));
#pragma unroll
      for (int e = 0; e < 8; ++e) asm volatile("" ::"v"(buf.v[e][0]), "v"(buf.v[e][1]));
      const TileLanes tl(lane);
      for (; p0 < P.end; p0 += STEP) {
        load_tile(buf, ks_s, tile_rsrc(kbase, p0, P.end, HD * 2),
                  tile_rsrc(vbase, p0, P.end, HD * 2), tl);
        wait_and_compute<NT>(buf, ks_lds, p0, P.Lmin, Lcol, qb, scale_log2, c, g4, m, l, acc);
      }
    } else {
      const TileLanes tl(lane);
      int p0 = P.beg + w * TILE;
      if (p0 < P.end) {
        uint32_t cur = ks_s, nxt = ks_s + TILE * HD * 2;  // two 16 KB slots
        issue_k(cur, tile_rsrc(kbase, p0, P.end, HD * 2), tl);
        __builtin_amdgcn_sched_barrier(0);
        issue_v(buf, tile_rsrc(vbase, p0, P.end, HD * 2), tl);
        for (; p0 + STEP < P.end; p0 += STEP) {
          vmcnt_wait<16>();  // this tile's K: its V (16 loads) may remain
          __builtin_amdgcn_sched_barrier(0);
          issue_k(nxt, tile_rsrc(kbase, p0 + STEP, P.end, HD * 2), tl);
          __builtin_amdgcn_sched_barrier(0);
          compute_tile<NT>(buf, lds_tile(cur), p0, P.Lmin, Lcol, qb, scale_log2, c, g4, m, l,
                           acc);
          __builtin_amdgcn_sched_barrier(0);
          issue_v(buf, tile_rsrc(vbase, p0 + STEP, P.end, HD * 2), tl);
          const uint32_t t = cur;
          cur = nxt;
          nxt = t;
        }
        vmcnt_wait<16>();
        compute_tile<NT>(buf, lds_tile(cur), p0, P.Lmin, Lcol, qb, scale_log2, c, g4, m, l, acc);
      }
    }

    // ---- merge the waves of this workgroup in a fixed order and write the slice's partial
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) l[ct] = group4_sum(l[ct]);

    static_assert(WAVES == 4, "merge layout assumes 4 waves");
    if constexpr (NT == 1) {
      // s_acc[v]: the first 16 KB of wave v's K slots
      auto s_acc = [&](int v, int a) __attribute__((always_inline)) -> f32x4_t& {
        return reinterpret_cast<f32x4_t*>(lds + v * WAREA)[a * WAVE + lane];
      };
      // One barrier: each wave parks (m, l) and the accumulators of the pass's columns in its own
      // K slots' LDS (s_acc(w, .) lies there, which no other wave touches), then thread
      // (w, lane) merges h = w/2, i in [4(w&1), +4) over waves 0..3 in that order and writes
      // 4 x 16 bytes: dims 128h + 32g4 + 8ii + 4(w&1) + [0, 4) for ii = 0..3. Same arithmetic
      // and order as the NT >= 2 merge below, so the bits do not depend on NT.
      const int col = c;
      const bool mine = in_pass(col, grp, P);
      // One tile: the other waves hold m = -inf, l = 0, O = 0, so wave 0's accumulators are the
      // partial, bit for bit, and no barrier is needed. A short prefix is a chain of latencies, and
      // the merge's two LDS passes were part of it: prep + decode of one row at 1k (24/4 heads)
      // went from 10.4 to 9.6 us. (Conditions on the number of active waves inside the general
      // sums, instead, put its LDS reads behind branches: 3% slower at 16k.)
      if (P.end - P.beg <= TILE) {
        if (w != 0 || !mine) return;
        const int t = trow[0], head = g * grp + (col - t * grp);
        const size_t slot = ((size_t)t * Hq + head) * NS + s;
        if (g4 == 0) {
          part_ml[slot * 2] = m[0];
          part_ml[slot * 2 + 1] = l[0];
        }
        float* dst = part_o + slot * HD + 32 * g4;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int ii = 0; ii < 4; ++ii)
#pragma unroll
            for (int i = 0; i < 8; i += 4)
              *reinterpret_cast<f32x4_t*>(dst + 128 * hh + 8 * ii + i) =
                  f32x4_t{acc[0][8 * hh + i][ii], acc[0][8 * hh + i + 1][ii],
                          acc[0][8 * hh + i + 2][ii], acc[0][8 * hh + i + 3][ii]};
        return;
      }
      if (g4 == 0) {
        s_m[w][col] = m[0];
        s_l[w][col] = l[0];
      }
      if (mine) {
#pragma unroll
        for (int a = 0; a < 16; ++a) s_acc(w, a) = acc[0][a];
      }
      lds_barrier();
      if (!mine) return;
      float M = -INFINITY, wsc[WAVES];
#pragma unroll
      for (int v = 0; v < WAVES; ++v) M = fmaxf(M, s_m[v][col]);
      float L = 0.f;
#pragma unroll
      for (int v = 0; v < WAVES; ++v) {
        const float mv = s_m[v][col];
        wsc[v] = mv == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mv - M);
        L += s_l[v][col] * wsc[v];
      }
      const int t = trow[0], head = g * grp + (col - t * grp);
      if (w == 0 && g4 == 0) {
        float* ml = part_ml + (((size_t)t * Hq + head) * NS + s) * 2;
        ml[0] = M;
        ml[1] = L;
      }
      const int h = w >> 1, i0 = 4 * (w & 1);
      f32x4_t mo[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < WAVES; ++v) sum += s_acc(v, 8 * h + i0 + k) * wsc[v];
        mo[k] = sum;
      }
      float* dst = part_o + (((size_t)t * Hq + head) * NS + s) * HD + 128 * h + 32 * g4 + i0;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii)
        reinterpret_cast<f32x4_t*>(dst + 8 * ii)[0] =
            f32x4_t{mo[0][ii], mo[1][ii], mo[2][ii], mo[3][ii]};
      return;
    }

    if (g4 == 0) {
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) {
        s_m[w][ct * 16 + c] = m[ct];
        s_l[w][ct * 16 + c] = l[ct];
      }
    }
    lds_barrier();  // also: every wave is done with its K tile, so `lds` can hold the merge

    float wsc[NT][WAVES];
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
      const int col = ct * 16 + c;
      float M = -INFINITY;
#pragma unroll
      for (int v = 0; v < WAVES; ++v) M = fmaxf(M, s_m[v][col]);
      float L = 0.f;
#pragma unroll
      for (int v = 0; v < WAVES; ++v) {
        const float mv = s_m[v][col];
        wsc[ct][v] = mv == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mv - M);
        L += s_l[v][col] * wsc[ct][v];
      }
      if (w == 0 && g4 == 0 && in_pass(col, grp, P)) {
        const int t = trow[ct], head = g * grp + (col - t * grp);
        float* ml = part_ml + (((size_t)t * Hq + head) * NS + s) * 2;
        ml[0] = M;
        ml[1] = L;
      }
    }

    // Each wave parks the O^T accumulators of the pass's columns in LDS as 16-byte rows (lanes of
    // other columns stay idle, which keeps the LDS traffic to what the merge needs), one barrier,
    // then thread (w, lane) merges h = w/2, i in [4(w&1), +4) over waves 0..3 in that order and
    // writes 4 x 16 bytes: dims 128h + 32g4 + 8ii + 4(w&1) + [0, 4) for ii = 0..3.
    f32x4_t (*s_acc)[16][WAVE] = reinterpret_cast<f32x4_t (*)[16][WAVE]>(lds);
    static_assert(WAVES * 16 * WAVE * 16 <= WAVES * WAREA, "merge buffer aliases the K tiles");
#pragma unroll
    for (int ct = 0; ct < NT; ++ct) {
      const int col = ct * 16 + c;
      const bool mine = in_pass(col, grp, P);
      if (ct > 0) lds_barrier();  // the previous column tile's reads are done (its stores need not be)
      if (mine) {
#pragma unroll
        for (int a = 0; a < 16; ++a) s_acc[w][a][lane] = acc[ct][a];
      }
      lds_barrier();
      if (mine) {
        const int h = w >> 1, i0 = 4 * (w & 1);
        f32x4_t mo[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int v = 0; v < WAVES; ++v) sum += s_acc[v][8 * h + i0 + k][lane] * wsc[ct][v];
          mo[k] = sum;
        }
        const int t = trow[ct], head = g * grp + (col - t * grp);
        float* dst = part_o + (((size_t)t * Hq + head) * NS + s) * HD + 128 * h + 32 * g4 + i0;
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
          reinterpret_cast<f32x4_t*>(dst + 8 * ii)[0] =
              f32x4_t{mo[0][ii], mo[1][ii], mo[2][ii], mo[3][ii]};
      }
    }
  };
  if (attendA) run_pass(PA, true);
  if constexpr (MULTI) {
    if (attendB) {
      if (attendA) lds_barrier();  // the merge's LDS reads are done before the next pass
      run_pass(PB, !attendA);
    }
  }
}

// Multi-row variant (NT >= 3 column tiles: six or more rows at GQA 6, up to 64 columns).
// A workgroup (slice, KV head) holds 4 position subsets x NT/CPW waves: wave (sub, rank) owns
// column tiles [rank*CPW, +CPW) for the slice's tiles k = sub (mod 4), the same tiles that wave
// `sub` of attn_partials_kernel processes, with the same per-column arithmetic, and the 4 subsets
// merge in the same order 0..3. So every column's partial is bit-identical to what the one-tile
// kernel computes for it, which keeps row t of an n-row call equal to a 1-row call. The waves of a
// subset share its K and V tile through LDS (LDS DMA, as in prefill); each wave keeps only its own
// columns' state in registers (<= 170 VGPRs at three waves per SIMD), where the one-tile kernel
// would need all NT column tiles per wave and spill.
namespace cols {
constexpr int SUBSETS = 4;
constexpr int TILE_U4 = TILE * ROW_CHUNKS;   // 16-byte slots of one K (or V) tile: 16 KB
constexpr int REGION_U4 = 2 * TILE_U4;       // a subset's K tile then V tile
}  // namespace cols

// Look-ahead rounds of attn_partials_cols_kernel. bf16 cache: round 0's K and V tiles load together;
// after that the V tile of round r loads while the subset computes S^T and the softmax of round r, and
// the K tile of round r+1 while it computes O^T += V^T P^T. fp8 cache, one column tile per wave: the fp8
// K tile of round r+1 loads into the subset's 8 KB staging buffer during S^T and the softmax of round r,
// is converted into the bf16 K tile, and the fp8 V tile of round r+1 then loads into the same buffer
// during O^T += V^T P^T. No operand read may wait for the loads just issued: on the fp8 cache each half
// takes its LDS operands and the LDS-DMA target as distinct __restrict__ pointers, on the bf16 cache the
// target is a plain LDS address (otherwise the compiler's wait-count pass waits for the loads before the
// first read).
namespace cols {
constexpr int STAGE8_U4 = TILE * HD / 16;  // 16-byte slots of one fp8 tile: 8 KB
// Operand reads kept ahead of the MFMAs in S^T and O^T. Same-box harness A/B at one column tile per wave,
// partials us, none -> 4: 5 rows at 4101 (config 3) 10.64 -> 10.42, 8 rows at 4104 13.45 -> 13.39, 8 rows
// at 16392 22.80 -> 22.49; bits identical. Two column tiles per wave on the fp8 cache spill and keep
// the compiler's order.
constexpr int LEAD = 4;

// 8 one-KB LDS-DMA loads of an fp8 tile, rows 4i .. 4i+3, row-major (chunk q of row r at 16 r + q)
__device__ __forceinline__ void issue_fp8(__amdgpu_buffer_rsrc_t rs, int p0, u32x4_t* dst, int rank,
                                          int wps, int lane) {
  for (int i = rank; i < 8; i += wps) {
    const int row = 4 * i + (lane >> 4);
    buffer_load16_to_lds(rs, (uint32_t)(p0 + row) * HD + (lane & 15) * 16, dst + 64 * i);
  }
}
// bf16 tiles of the bf16-cache kernels: rows in pairs of 1024 bytes plus a pad, row 2p + o at
// PAIR p + 512 o. K's 16-byte chunks are XORed with o and V's 32-byte pieces with o, which spreads
// the 16 rows of a K read and the 8 rows of a transposing V read over all banks with every address
// one (K) or two (V) per-lane bases plus an immediate. (The XOR by row & 15 of tile::k_slot needs an
// address per read, and with two column tiles a wave has no registers for them.)
constexpr int KPAIR = 2 * HD * 2 + 32, VPAIR = 2 * HD * 2 + 64;
constexpr int KTILE_P = TILE / 2 * KPAIR, REGION_P = KTILE_P + TILE / 2 * VPAIR;  // bytes
// 16 one-KB LDS-DMA loads (a row pair each) of a bf16 K (or V) tile, shared by the subset's waves.
// rs starts at the tile's first row. dst, the tile's LDS byte address, and rank, the wave in the subset,
// are in scalar registers, so that M0 is scalar arithmetic. The lane offsets are made anew for every
// tile (opaque to the compiler): hoisted out of the rounds they are a register per load, which the
// kernel of two column tiles per wave has to spill, and the reload of a spilled offset waits for the
// load before it. us per call, loop without look-ahead / offsets hoisted (41 VGPRs spilled) / now (none): 8
// rows at 16 / 2 heads on 6k 25.0 / 22.8 / 22.5, 16k 31.4 / 33.6 / 26.8, 64k 52.2 / 64.9 / 42.4; three column
// tiles, 8 rows at 24 / 4 on 64k 60.2 / 60.8 / 57.2. (The pair's place is not in the instruction's scalar
// offset, which the range check leaves out.)
template <bool IS_V, int WPS>
__device__ __forceinline__ void issue_pairs(__amdgpu_buffer_rsrc_t rs, uint32_t dst, int rank, int lane) {
  const uint32_t o = lane >> 5;
  uint32_t off = o * (HD * 2) + ((lane & 31) ^ (IS_V ? 2 * o : o)) * 16 + rank * (2 * HD * 2);
  asm volatile("" : "+v"(off));
  dst += rank * (IS_V ? VPAIR : KPAIR);
#pragma unroll
  for (int k = 0; k < (16 + WPS - 1) / WPS; ++k)
    if (16 % WPS == 0 || k * WPS + rank < 16)
      buffer_load16_to_lds_at(rs, off + k * (WPS * 2 * HD * 2), dst + k * (WPS * (IS_V ? VPAIR : KPAIR)));
}
// S^T of a tile, tile::qk_tile's arithmetic: operand k = positions 16 (k >> 3) .., dims 32 (k & 7) ..;
// LEAD reads run ahead of the MFMAs.
template <int CPW>
__device__ __forceinline__ void qk_pairs(const char* __restrict__ kt, const bf16x8_t (&qb)[CPW][8],
                                         int lane, f32x4_t (&sacc)[CPW][2]) {
  const int c = lane & 15, o = c & 1;
  const char* k0 = kt + (c >> 1) * KPAIR + o * (HD * 2) + 16 * ((lane >> 4) ^ o);
  auto read = [&](int k) __attribute__((always_inline)) {
    return as_bf16x8(*reinterpret_cast<const u32x4_t*>(k0 + (k >> 3) * (8 * KPAIR) + 64 * (k & 7)));
  };
  bf16x8_t op[16];
#pragma unroll
  for (int k = 0; k < LEAD; ++k) op[k] = read(k);
#pragma unroll
  for (int u = 0; u < CPW; ++u) sacc[u][0] = sacc[u][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < 16; ++k) {
#pragma unroll
    for (int u = 0; u < CPW; ++u) sacc[u][k >> 3] = mfma16x16x32(op[k], qb[u][k & 7], sacc[u][k >> 3]);
    if (k + LEAD < 16) op[k + LEAD] = read(k + LEAD);
    __builtin_amdgcn_sched_barrier(0);
  }
}
// O^T += V^T P^T of a tile, tile::pv_tile_tr's arithmetic (P as hi + lo terms).
template <int CPW>
__device__ __forceinline__ void pv_pairs(const char* __restrict__ vt, int lane,
                                         const u32x4_t (&hi)[CPW], const u32x4_t (&lo)[CPW],
                                         f32x4_t (&acc)[CPW][16]) {
  typedef short v4i16 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4i16 lds_v4i16;
  const int x = (lane >> 2) & 3, o = x & 1;  // rows 4 g4 + x and + 16, dims 16i + 4 (lane & 3) .. +3
  const char* v0 = vt + (2 * (lane >> 4) + (x >> 1)) * VPAIR + o * (HD * 2) + 8 * (lane & 3);
  const char* vb[2] = {v0 + 32 * o, v0 + 32 * (1 - o)};  // piece i of the row is at i ^ o
  auto read = [&](int i) __attribute__((always_inline)) {
    const char* a = vb[i & 1] + 32 * (i & 14);
    const u32x2_t y = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)a));
    const u32x2_t z = __builtin_bit_cast(
        u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(a + 8 * VPAIR)));
    return as_bf16x8(u32x4_t{y[0], y[1], z[0], z[1]});
  };
  bf16x8_t op[16];
#pragma unroll
  for (int i = 0; i < LEAD; ++i) op[i] = read(i);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
      acc[u][i] = mfma16x16x32(op[i], as_bf16x8(hi[u]), acc[u][i]);
      acc[u][i] = mfma16x16x32(op[i], as_bf16x8(lo[u]), acc[u][i]);
    }
    if (i + LEAD < 16) op[i + LEAD] = read(i + LEAD);
    __builtin_amdgcn_sched_barrier(0);
  }
}
template <int CPW>
__device__ __forceinline__ void softmax(const f32x4_t (&sacc)[CPW][2], int p0, int Lmin,
                                        const int (&Lcol)[CPW], float scale_log2, int g4,
                                        float (&m)[CPW], float (&l)[CPW], f32x4_t (&acc)[CPW][16],
                                        u32x4_t (&pb_hi)[CPW], u32x4_t (&pb_lo)[CPW]) {
  if (p0 + TILE > Lmin)
    tile::softmax_tile<CPW, true, true>(sacc, p0, Lcol, scale_log2, g4, m, l, acc, pb_hi, pb_lo);
  else
    tile::softmax_tile<CPW, false, true>(sacc, p0, Lcol, scale_log2, g4, m, l, acc, pb_hi, pb_lo);
}
// The two halves of a look-ahead round on the bf16 cache: what one half loads is never what it reads.
template <int CPW, int WPS>
__device__ __forceinline__ void half_s(const char* __restrict__ kt, uint32_t vt, bool has,
                                       bool load, __amdgpu_buffer_rsrc_t vrs, int p0, int Lmin,
                                       int rank, int lane, const bf16x8_t (&qb)[CPW][8],
                                       const int (&Lcol)[CPW], float scale_log2, float (&m)[CPW],
                                       float (&l)[CPW], f32x4_t (&acc)[CPW][16],
                                       u32x4_t (&pb_hi)[CPW], u32x4_t (&pb_lo)[CPW]) {
  if (load) issue_pairs<true, WPS>(vrs, vt, rank, lane);
  if (!has) return;
  f32x4_t sacc[CPW][2];
  qk_pairs<CPW>(kt, qb, lane, sacc);
  softmax<CPW>(sacc, p0, Lmin, Lcol, scale_log2, lane >> 4, m, l, acc, pb_hi, pb_lo);
}
template <int CPW, int WPS>
__device__ __forceinline__ void half_o(const char* __restrict__ vt, uint32_t kt, bool has,
                                       bool load, __amdgpu_buffer_rsrc_t krs, int rank, int lane, const u32x4_t (&pb_hi)[CPW],
                                       const u32x4_t (&pb_lo)[CPW], f32x4_t (&acc)[CPW][16]) {
  if (load) issue_pairs<false, WPS>(krs, kt, rank, lane);
  if (has) pv_pairs<CPW>(vt, lane, pb_hi, pb_lo, acc);
}
// The fp8 cache's halves: each loads an fp8 tile into the staging buffer.
template <int CPW>
__device__ __forceinline__ void qk_softmax_half(
    const u32x4_t* __restrict__ kt, u32x4_t* __restrict__ dst, bool has, bool load, int p_load,
    __amdgpu_buffer_rsrc_t rs, int p0, int Lmin, int rank, int wps, int lane, int c, int g4,
    const bf16x8_t (&qb)[CPW][8], const int (&Lcol)[CPW], float scale_log2, float (&m)[CPW],
    float (&l)[CPW], f32x4_t (&acc)[CPW][16], u32x4_t (&pb_hi)[CPW], u32x4_t (&pb_lo)[CPW]) {
  if (load) issue_fp8(rs, p_load, dst, rank, wps, lane);
  if (!has) return;
  f32x4_t sacc[CPW][2];
  tile::qk_tile<CPW, false, LEAD>(kt, qb, c, g4, sacc);
  softmax<CPW>(sacc, p0, Lmin, Lcol, scale_log2, g4, m, l, acc, pb_hi, pb_lo);
}
template <int CPW>
__device__ __forceinline__ void pv_half_la(const u32x4_t* __restrict__ vt,
                                           u32x4_t* __restrict__ dst, bool has, bool load,
                                           int p_load, __amdgpu_buffer_rsrc_t rs, int rank,
                                           int wps, int lane, int g4,
                                           const u32x4_t (&pb_hi)[CPW], const u32x4_t (&pb_lo)[CPW],
                                           f32x4_t (&acc)[CPW][16]) {
  if (load) issue_fp8(rs, p_load, dst, rank, wps, lane);
  if (has) tile::pv_tile_tr<CPW, true, false, LEAD>(vt, lane, g4, pb_hi, pb_lo, acc);
}
// All NTH threads of the workgroup convert the fp8 tiles of the first nact subsets once, from
// `src` (row-major) to `dst` (the bf16 K or V tile layout) in each subset's region of `region`
// slots. Every E4M3 value is a bf16 value, so the conversion is exact.
template <bool IS_V, int NTH>
__device__ __forceinline__ void convert_fp8(u32x4_t* lds, int region, int src_off, int dst_off,
                                            int nact) {
  constexpr int IT = (SUBSETS * STAGE8_U4 + NTH - 1) / NTH;
  int tid = threadIdx.x;  // opaque: the slot arithmetic is redone at each call
  asm volatile("" : "+v"(tid));
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int gk = it * NTH + tid;
    if (gk < nact * STAGE8_U4) {  // uniform per wave
      const int ss = gk / STAGE8_U4, i = gk % STAGE8_U4, rr = i >> 4, q = i & 15;
      u32x4_t* base = lds + ss * region;
      const u32x4_t c8 = base[src_off + i];
      const u32x4_t lo = fp8x8_to_bf16x8(u32x2_t{c8[0], c8[1]});
      const u32x4_t hi = fp8x8_to_bf16x8(u32x2_t{c8[2], c8[3]});
      if constexpr (IS_V) {
        base[dst_off + rr * ROW_CHUNKS + ((2 * q) ^ tile::v_swz(rr))] = lo;
        base[dst_off + rr * ROW_CHUNKS + ((2 * q + 1) ^ tile::v_swz(rr))] = hi;
      } else {
        base[dst_off + tile::k_slot(rr, 2 * q)] = lo;
        base[dst_off + tile::k_slot(rr, 2 * q + 1)] = hi;
      }
    }
  }
}
}  // namespace cols

// KV8: an fp8 cache (E4M3FN codes). The subset's 8 KB fp8 K and V tiles land row-major in LDS
// and all waves of the workgroup convert each tile once (exactly: every E4M3 value is a bf16
// value) into the bf16 K and V tiles, laid out and swizzled as the bf16 path loads them, so the
// tile arithmetic runs unchanged. With scales of 1 the result equals the bf16 kernel's on the
// dequantized cache, bit for bit. Converting once instead of in every wave that reads a tile took
// the 8-row verify from 17.1 to 14.7 us (partials, 4k) and 29.0 to 25.0 (16k); the look-ahead
// rounds (one column tile per wave: a staging buffer per subset, 160 KB of LDS) then took it to
// 13.7 (4k), 21.6 (16k) and 30.2 (32k). With two column tiles per wave the fp8 tiles of a round
// land in the subset's 16 KB V tile (K, then V) and are converted before its arithmetic.
template <int NT, int CPW, bool KV8 = false>
__global__ void __launch_bounds__(cols::SUBSETS * (NT / CPW) * WAVE)
attn_partials_cols_kernel(const __bf16* __restrict__ q, const __bf16* __restrict__ kc,
                          const __bf16* __restrict__ vc, const int* __restrict__ pos_ptr,
                          float* __restrict__ part_o, float* __restrict__ part_ml, int n, int Hq,
                          int Hkv, int max_len, int NS, NsDiv nd, float scale_log2, int row0) {
  static_assert(NT % CPW == 0, "column tiles split evenly over the waves of a subset");
  constexpr int SUB = cols::SUBSETS;
  constexpr int WPS = NT / CPW;  // waves per subset
  const int pos0 = pos_ptr[0] + row0;  // first: the slicing waits for it
  asm volatile("" ::: "memory");       // (and it is not sunk below the query's loads)
  const int s = blockIdx.x, g = blockIdx.y;
  const int grp = Hq / Hkv;
  const int lane = threadIdx.x & (WAVE - 1);
  const int w = KV8 ? (int)(threadIdx.x / WAVE) : __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  // A subset's waves are consecutive, so that slices with fewer tiles than subsets still spread over
  // the SIMDs (wave w runs on SIMD w mod 4).
  const int sub = w / WPS, rank = w % WPS;
  const int c = lane & 15, g4 = lane >> 4;
  const int ncols = grp * n;

  bf16x8_t qb[CPW][8];  // loaded before pos arrives (it does not depend on it)
#pragma unroll
  for (int u = 0; u < CPW; ++u) {
    const int col = (rank * CPW + u) * 16 + c;
    if (col < ncols) {
      const int t = col / grp, j = col - t * grp;
      const u32x4_t* src =
          reinterpret_cast<const u32x4_t*>(q + (size_t)t * Hq * HD + (size_t)(g * grp + j) * HD);
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) qb[u][ks] = as_bf16x8(src[4 * ks + g4]);
    } else {
#pragma unroll
      for (int ks = 0; ks < 8; ++ks) qb[u][ks] = as_bf16x8(u32x4_t{0u, 0u, 0u, 0u});
    }
  }

  int ch0, tB;
  call_split(pos0, n, max_len, NS, nd, ch0, tB);
  const int npass = tB < n ? 2 : 1;
  const Pass PA = pass_of(0, ch0, tB, n, pos0, max_len, s);
  const Pass PB = pass_of(1, ch0, tB, n, pos0, max_len, s);
  const bool attendA = PA.beg < PA.end;
  if (!attendA && !(npass > 1 && PB.beg < PB.end)) return;  // uniform per workgroup

  // fp8 with one column tile per wave: each subset's region also holds an 8 KB fp8 staging
  // buffer (4 x 40 KB: all 160 KB of LDS), and s_m / s_l live in the ring past the merge's two
  // accumulator buffers (the ring is idle once the rounds end).
  constexpr bool LA8 = KV8 && CPW == 1;
  constexpr int REGION = !KV8 ? cols::REGION_P / 16 : LA8 ? cols::REGION_U4 + cols::STAGE8_U4 : cols::REGION_U4;
  __shared__ __attribute__((aligned(16))) u32x4_t lds[SUB * REGION];  // 134 KB (bf16), 128 or 160 KB
  __shared__ float s_m_[LA8 ? 1 : SUB][16 * NT], s_l_[LA8 ? 1 : SUB][16 * NT];
  static_assert(!LA8 || 2 * SUB * 16 * WAVE * 16 + 2 * SUB * 16 * NT * 4 <= SUB * REGION * 16,
                "s_m and s_l fit the ring past the two merge buffers");
  float (*s_m)[16 * NT] =
      LA8 ? reinterpret_cast<float (*)[16 * NT]>(lds + 2 * SUB * 16 * WAVE) : s_m_;
  float (*s_l)[16 * NT] =
      LA8 ? reinterpret_cast<float (*)[16 * NT]>(lds + 2 * SUB * 16 * WAVE) + SUB : s_l_;
  constexpr int ELEM = KV8 ? 1 : 2;  // bytes per cache value
  const size_t head_off = (size_t)g * max_len * HD * ELEM;  // bytes
  u32x4_t* kt = lds + sub * REGION;
  u32x4_t* vt = kt + cols::TILE_U4;
  u32x4_t* st = vt + cols::TILE_U4;  // LA8: the fp8 staging buffer
  char *kp = reinterpret_cast<char*>(kt), *vp = kp + cols::KTILE_P;  // bf16 cache
  const uint32_t kl = KV8 ? 0 : lds_byte_uniform(kt);

  // One pass, inlined once per call of the lambda (a loop over passes would keep the merge's
  // loop-invariant addresses live through the tile rounds and spill).
  auto run_pass = [&](const Pass P, bool more) __attribute__((always_inline)) {
    // The columns' attended lengths, computed once the first tile's loads are out: what is reloaded
    // for them (the registers are few) waits for every load before it, the query's first of all.
    int Lcol[CPW];
    auto lcol = [&]() __attribute__((always_inline)) {
      int cc = c;
      asm volatile("" : "+v"(cc));
#pragma unroll
      for (int u = 0; u < CPW; ++u)
        Lcol[u] = in_pass((rank * CPW + u) * 16 + cc, grp, P)
                      ? min(pos0 + ((rank * CPW + u) * 16 + cc) / grp + 1, max_len) : 0;
    };
    // fp8 cache: the KV head's rows up to the pass's end
    const auto head_rsrc = [&](const __bf16* base) __attribute__((always_inline)) {
      return make_rsrc_uniform(reinterpret_cast<const char*>(base) + head_off,
                               (uint32_t)P.end * (uint32_t)(HD * ELEM));
    };

    float m[CPW], l[CPW];
    f32x4_t acc[CPW][16];  // tile::pv_tile_tr layout
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
      m[u] = -INFINITY;
      l[u] = 0.f;
#pragma unroll
      for (int a = 0; a < 16; ++a) acc[u][a] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    const int ntiles = (P.end - P.beg + TILE - 1) / TILE;
    const int rounds = (ntiles + SUB - 1) / SUB;
    if constexpr (!KV8) {
      // Two barriers per round (one when the pass has one round); each one also publishes the tile
      // loaded during the half-round before it.
      const auto rsrc = [&](const __bf16* base, int p) __attribute__((always_inline)) {
        return tile_rsrc(reinterpret_cast<const char*>(base) + head_off, p, P.end, HD * 2);
      };
      const int p00 = P.beg + sub * TILE;
      if (p00 < P.end) {
        cols::issue_pairs<false, WPS>(rsrc(kc, p00), kl, rank, lane);
        cols::issue_pairs<true, WPS>(rsrc(vc, p00), kl + cols::KTILE_P, rank, lane);
      }
      lcol();
      vmcnt_wait<0>();
      __syncthreads();  // K and V of round 0 have landed
      for (int r = 0; r < rounds; ++r) {
        const int p0 = P.beg + (r * SUB + sub) * TILE;  // this subset's tile in round r
        const bool has = p0 < P.end;                     // uniform per subset
        const int p1 = p0 + SUB * TILE;
        const bool has1 = r + 1 < rounds && p1 < P.end;
        u32x4_t pb_hi[CPW], pb_lo[CPW];
        cols::half_s<CPW, WPS>(kp, kl + cols::KTILE_P, has, has && r > 0, rsrc(vc, p0), p0, P.Lmin, rank,
                               lane, qb, Lcol, scale_log2, m, l, acc, pb_hi, pb_lo);
        // (The wait stays outside the branch: behind a join the compiler's wait-count pass
        // assumes V may still be in flight and waits for the K load below before PV.)
        vmcnt_wait<0>();
        if (r > 0 || r + 1 < rounds)  // uniform
          __syncthreads();  // V of round r has landed; K of round r is no longer read
        cols::half_o<CPW, WPS>(vp, kl, has, has1, rsrc(kc, p1), rank, lane, pb_hi, pb_lo, acc);
        vmcnt_wait<0>();
        __syncthreads();  // K of round r+1 has landed; V of round r is no longer read
      }
    } else if constexpr (LA8) {
      const __amdgpu_buffer_rsrc_t krs = head_rsrc(kc), vrs = head_rsrc(vc);
      constexpr int NTH = SUB * WPS * WAVE;
      const auto nact = [&](int r) {  // active subsets of round r (>= 1 for r < rounds)
        return min(SUB, (P.end - (P.beg + r * SUB * TILE) + TILE - 1) / TILE);
      };
      // Round 0: fp8 K into the staging buffer and fp8 V into the upper half of the bf16 K tile,
      // together; V is converted first, then K over the slots V came from.
      const int p00 = P.beg + sub * TILE;
      if (p00 < P.end) {
        cols::issue_fp8(krs, p00, st, rank, WPS, lane);
        cols::issue_fp8(vrs, p00, kt + cols::STAGE8_U4, rank, WPS, lane);
      }
      lcol();
      vmcnt_wait<0>();
      __syncthreads();  // the fp8 tiles of round 0 have landed
      cols::convert_fp8<true, NTH>(lds, REGION, cols::STAGE8_U4, cols::TILE_U4, nact(0));
      __syncthreads();  // bf16 V whole; its fp8 source is no longer read
      cols::convert_fp8<false, NTH>(lds, REGION, 2 * cols::TILE_U4, 0, nact(0));
      __syncthreads();  // bf16 K whole; the staging buffer is free
      for (int r = 0; r < rounds; ++r) {
        const int p0 = P.beg + (r * SUB + sub) * TILE;  // this subset's tile in round r
        const bool has = p0 < P.end;                     // uniform per subset
        const int p1 = p0 + SUB * TILE;
        const bool more = r + 1 < rounds;                // uniform
        const bool has1 = more && p1 < P.end;
        u32x4_t pb_hi[CPW], pb_lo[CPW];
        cols::qk_softmax_half<CPW>(kt, st, has, has1, p1, krs, p0, P.Lmin, rank, WPS, lane, c,
                                      g4, qb, Lcol, scale_log2, m, l, acc, pb_hi, pb_lo);
        // (The waits stay outside the branches: behind a join the compiler's wait-count pass
        // would assume a load in flight and wait for the next one before the operand reads.)
        vmcnt_wait<0>();
        if (more) {
          __syncthreads();  // fp8 K of round r+1 has landed; bf16 K of round r is no longer read
          cols::convert_fp8<false, NTH>(lds, REGION, 2 * cols::TILE_U4, 0, nact(r + 1));
          __syncthreads();  // bf16 K of round r+1 whole; the staging buffer is free
        }
        cols::pv_half_la<CPW>(vt, st, has, has1, p1, vrs, rank, WPS, lane, g4, pb_hi, pb_lo,
                                 acc);
        vmcnt_wait<0>();
        __syncthreads();  // fp8 V of round r+1 has landed; bf16 V of round r is no longer read
        if (more) {
          cols::convert_fp8<true, NTH>(lds, REGION, 2 * cols::TILE_U4, cols::TILE_U4, nact(r + 1));
          __syncthreads();  // bf16 V of round r+1 whole; the staging buffer is free
        }
      }
    } else {  // fp8 cache, two column tiles per wave: no look-ahead (no registers for it)
      const __amdgpu_buffer_rsrc_t krs = head_rsrc(kc), vrs = head_rsrc(vc);
      for (int r = 0; r < rounds; ++r) {
        if (r == 0) lcol();
        const int p0 = P.beg + (r * SUB + sub) * TILE;  // this subset's tile in round r
        const bool has = p0 < P.end;                     // uniform per subset
        if (has) {
          // fp8: 8 loads of K then 8 of V, one KB (rows 4j .. 4j+3) each, shared by the subset's
          // waves: 16-byte chunk q of row r of K at vt[16 r + q], of V at vt[512 + 16 r + q].
          for (int i = rank; i < 16; i += WPS) {
            const int row = 4 * (i & 7) + (lane >> 4);
            buffer_load16_to_lds(i < 8 ? krs : vrs, (uint32_t)(p0 + row) * HD + (lane & 15) * 16,
                                 vt + 64 * i);
          }
        }
        vmcnt_wait<0>();
        __syncthreads();  // every wave's loads of this round have landed
        // Convert once, all waves of the workgroup together: chunk gk of the active subsets'
        // tiles (subset gk / 512, chunk gk % 512) goes to thread gk % (64 SUB WPS).
        constexpr int CHUNKS = TILE * HD / 16;  // 16-byte fp8 chunks per tile
        constexpr int NTH = SUB * WPS * WAVE;
        constexpr int IT = (SUB * CHUNKS + NTH - 1) / NTH;
        const int rem = P.end - (P.beg + r * SUB * TILE);
        const int nact = min(SUB, (rem + TILE - 1) / TILE);  // active subsets this round (>= 1)
        u32x4_t v8[IT];
        int tid = threadIdx.x;  // opaque: the slot arithmetic is redone each round
        asm volatile("" : "+v"(tid));
#pragma unroll
        for (int it = 0; it < IT; ++it) {
          const int gk = it * NTH + tid;
          if (gk < nact * CHUNKS) {  // uniform per wave
            const int ss = gk / CHUNKS, i = gk % CHUNKS, rr = i >> 4, q = i & 15;
            u32x4_t* kts = lds + ss * cols::REGION_U4;
            const u32x4_t* vts = kts + cols::TILE_U4;
            v8[it] = vts[CHUNKS + i];
            const u32x4_t k8 = vts[i];
            kts[tile::k_slot(rr, 2 * q)] = fp8x8_to_bf16x8(u32x2_t{k8[0], k8[1]});
            kts[tile::k_slot(rr, 2 * q + 1)] = fp8x8_to_bf16x8(u32x2_t{k8[2], k8[3]});
          }
        }
        __syncthreads();  // the bf16 K tiles are whole, and no fp8 chunk is read again
#pragma unroll
        for (int it = 0; it < IT; ++it) {
          const int gk = it * NTH + tid;
          if (gk < nact * CHUNKS) {
            const int ss = gk / CHUNKS, i = gk % CHUNKS, rr = i >> 4, q = i & 15;
            u32x4_t* vts = lds + ss * cols::REGION_U4 + cols::TILE_U4;
            vts[rr * ROW_CHUNKS + ((2 * q) ^ tile::v_swz(rr))] =
                fp8x8_to_bf16x8(u32x2_t{v8[it][0], v8[it][1]});
            vts[rr * ROW_CHUNKS + ((2 * q + 1) ^ tile::v_swz(rr))] =
                fp8x8_to_bf16x8(u32x2_t{v8[it][2], v8[it][3]});
          }
        }
        __builtin_amdgcn_sched_barrier(0);  // keep the K operand reads below the conversion
        f32x4_t sacc[CPW][2];
        u32x4_t pb_hi[CPW], pb_lo[CPW];
        if (has) {
          tile::qk_tile<CPW, false, 0>(kt, qb, c, g4, sacc);
          if (p0 + TILE > P.Lmin)
            tile::softmax_tile<CPW, true, true>(sacc, p0, Lcol, scale_log2, g4, m, l, acc, pb_hi, pb_lo);
          else
            tile::softmax_tile<CPW, false, true>(sacc, p0, Lcol, scale_log2, g4, m, l, acc, pb_hi, pb_lo);
        }
        __syncthreads();  // the bf16 V tile is whole
        if (has) tile::pv_tile_tr<CPW, true, false, 0>(vt, lane, g4, pb_hi, pb_lo, acc);
        __syncthreads();  // this round's tiles are read before the next round overwrites them
      }
    }

    // ---- merge the 4 subsets in order 0..3 (as attn_partials_kernel merges its waves). Subsets
    // without a tile hold m = -inf, l = 0, O = 0: with at most two tiles the terms of subsets 2 and 3
    // (weight 0) stay out, which changes no bit. The barriers order LDS alone, not the stores.
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
      l[u] = group4_sum(l[u]);
      if (g4 == 0) {
        s_m[sub][(rank * CPW + u) * 16 + c] = m[u];
        s_l[sub][(rank * CPW + u) * 16 + c] = l[u];
      }
    }
    lds_barrier();
    float wsc[CPW][SUB];
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
      const int col = (rank * CPW + u) * 16 + c;
      float M = -INFINITY;
#pragma unroll
      for (int v = 0; v < SUB; ++v) M = fmaxf(M, s_m[v][col]);
      float L = 0.f;
#pragma unroll
      for (int v = 0; v < SUB; ++v) {
        const float mv = s_m[v][col];
        wsc[u][v] = mv == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mv - M);
        L += s_l[v][col] * wsc[u][v];
      }
      if (sub == 0 && g4 == 0 && in_pass(col, grp, P)) {
        const int t = col / grp, head = g * grp + (col - t * grp);
        float* ml = part_ml + (((size_t)t * Hq + head) * NS + s) * 2;
        ml[0] = M;
        ml[1] = L;
      }
    }
    // The (rank, column tile) items are merged two at a time: each item's accumulators from the 4
    // subsets take 64 KB, and two fill the ring, so one barrier pair serves both (3-4 rows at
    // GQA 6: all of them). Thread (sub, lane) of an item's owner rank merges accumulators
    // 4 sub .. 4 sub + 3 over the subsets in order 0..3.
    constexpr int GROUP = 2;
    constexpr int NI = WPS * CPW;  // items, rank-major within each column tile u
    static_assert(GROUP * SUB * 16 * WAVE * 16 <= SUB * cols::REGION_U4 * 16,
                  "two items' merge buffers fit the ring");
    f32x4_t (*s_acc)[SUB][16][WAVE] = reinterpret_cast<f32x4_t (*)[SUB][16][WAVE]>(lds);
    auto merge = [&](auto na) __attribute__((always_inline)) {
      constexpr int NA = decltype(na)::value;
#pragma unroll
      for (int i0 = 0; i0 < NI; i0 += GROUP) {
#pragma unroll
        for (int gi = 0; gi < GROUP; ++gi) {
          if (i0 + gi >= NI) break;
          const int u = (i0 + gi) / WPS, rr = (i0 + gi) % WPS;
          if (rank == rr && sub < NA && in_pass((rr * CPW + u) * 16 + c, grp, P)) {
#pragma unroll
            for (int a = 0; a < 16; ++a) s_acc[gi][sub][a][lane] = acc[u][a];
          }
        }
        lds_barrier();
#pragma unroll
        for (int gi = 0; gi < GROUP; ++gi) {
          if (i0 + gi >= NI) break;
          const int u = (i0 + gi) / WPS, rr = (i0 + gi) % WPS;
          const int col = (rr * CPW + u) * 16 + c;
          if (rank == rr && in_pass(col, grp, P)) {
            f32x4_t mo[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int v = 0; v < NA; ++v) sum += s_acc[gi][v][4 * sub + k][lane] * wsc[u][v];
              mo[k] = sum;
            }
            const int t = col / grp, head = g * grp + (col - t * grp);
            float* dst = part_o + (((size_t)t * Hq + head) * NS + s) * HD;
            // acc[i][k] = O^T[16i + 4g4 + k] (tile::pv_tile_tr)
#pragma unroll
            for (int k = 0; k < 4; ++k)
              reinterpret_cast<f32x4_t*>(dst + 16 * (4 * sub + k) + 4 * g4)[0] = mo[k];
          }
        }
        if (more || i0 + GROUP < NI) lds_barrier();  // (also ends the pass: the next one loads over `lds`)
      }
    };
    if (CPW == 1 && ntiles <= 2)
      merge(std::integral_constant<int, 2>{});
    else
      merge(std::integral_constant<int, SUB>{});
  };
  const bool attendB = npass > 1 && PB.beg < PB.end;
  if (attendA) run_pass(PA, attendB);
  if (attendB) run_pass(PB, false);
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

static hipError_t check_decode_shape(int n, int Hq, int Hkv, int max_len, int NS) {
  if (n < 1 || n > MAX_DECODE_ROWS || Hq < 1 || Hkv < 1 || Hq % Hkv != 0 || NS < 1 ||
      max_len < 1)
    return hipErrorInvalidValue;
  // byte offsets of the last tile (up to one tile past max_len) must fit the 32-bit buffer range
  if ((unsigned long long)(max_len + TILE) * HD * 2 >= (1ull << 32))
    return hipErrorInvalidValue;
  return hipSuccess;
}

// One launch of the partials kernels: n <= 8 rows and at most 64 query columns per workgroup
// ((Hq/Hkv) n <= 64, 4 tiles of 16), the first row at position pos[0] + row0. kv8: the cache is the fp8 KV format; k_scale multiplies
// every score (q . (code * k_scale)), folded into the softmax scale.
static hipError_t launch_partials_tiles(const void* q, const void* kc, const void* vc,
                                        const int* pos, float* part_o, float* part_ml, int n,
                                        int Hq, int Hkv, int max_len, int NS, float scale,
                                        hipStream_t stream, bool kv8, float k_scale, int row0) {
  const dim3 grid(max_slices(max_len, NS), Hkv);
  const NsDiv nd = ns_div(NS);
  const float scale_log2 = scale * 1.4426950408889634f * k_scale;
  const int NT = ((Hq / Hkv) * n + 15) / 16;
  const auto* Q = static_cast<const __bf16*>(q);
  const auto* K = static_cast<const __bf16*>(kc);
  const auto* V = static_cast<const __bf16*>(vc);
  if (kv8) {
    if (NT == 1 && n == 1)
      attn_partials_kernel<1, false, false, true><<<grid, dim3(waves_for<1>() * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, PrepIn{}, row0);
    else if (NT == 1)
      attn_partials_kernel<1, false, true, true><<<grid, dim3(waves_for<1>() * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, PrepIn{}, row0);
    else if (NT == 2)
      attn_partials_kernel<2, false, true, true><<<grid, dim3(waves_for<2>() * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, PrepIn{}, row0);
    else if (NT == 3)
      attn_partials_cols_kernel<3, 1, true><<<grid, dim3(cols::SUBSETS * 3 * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, row0);
    else
      attn_partials_cols_kernel<4, 2, true><<<grid, dim3(cols::SUBSETS * 2 * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, row0);
    return hipGetLastError();
  }
  // NT = 1, 2: every wave holds all column tiles (measured fastest at 1-5 rows, GQA 6), except
  // NT = 2 on caches whose slices hold at most 4 tiles (max_len <= 128 NS): there the 4 waves of
  // attn_partials_kernel<2> leave half the CU idle, and the multi-column kernel (one column tile
  // per wave, 8 waves) measured 7-10% faster at 4k-8k (it is 3-10% slower on 8-16-tile slices).
  // The two give the same bits per column.
  // NT = 3, 4: one subset wave per column tile (the one-tile kernel would spill: 2.3-2.8x slower).
  if (NT == 2 && split_size(max_len, nd) <= 4 * TILE) {
    attn_partials_cols_kernel<2, 1><<<grid, dim3(cols::SUBSETS * 2 * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, row0);
    return hipGetLastError();
  }
  switch (NT) {
    case 1:
      if (n == 1)
        attn_partials_kernel<1, false, false><<<grid, dim3(waves_for<1>() * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, PrepIn{}, row0);
      else
        attn_partials_kernel<1><<<grid, dim3(waves_for<1>() * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, PrepIn{}, row0);
      break;
    case 2: attn_partials_kernel<2><<<grid, dim3(waves_for<2>() * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, PrepIn{}, row0); break;
    case 3: attn_partials_cols_kernel<3, 1><<<grid, dim3(cols::SUBSETS * 3 * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, row0); break;
    default: attn_partials_cols_kernel<4, 2><<<grid, dim3(cols::SUBSETS * 2 * WAVE), 0, stream>>>(Q, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, row0); break;
  }
  return hipGetLastError();
}

// Any row count and group size, as several launches of the kernels above when one launch's 64
// query columns do not hold the call. Rows are independent (row t attends up to position
// pos[0] + t, reads q[t] and writes part_o[t], part_ml[t]), so a chunk of rows starting at row
// r0 is the same call on offset q / part_o / part_ml pointers with row0 = r0. Up to 64 q
// heads per KV head (G = Hq/Hkv), chunks of min(8, 64/G) rows. Beyond that, one row per launch
// and each KV head's q heads in ceil(G/64) sub-groups of consecutive heads, each launched as a
// one-KV-head call (Hkv = 1) on that head's cache and the sub-group's q, part_o and part_ml
// heads. A column's arithmetic does not depend on how many columns its launch holds, so every
// row of every shape has the bits of a 1-row call.
static hipError_t launch_partials(const void* q, const void* kc, const void* vc, const int* pos,
                                  float* part_o, float* part_ml, int n, int Hq, int Hkv,
                                  int max_len, int NS, float scale, hipStream_t stream,
                                  bool kv8 = false, float k_scale = 1.f) {
  const int G = Hq / Hkv;
  const auto* Q = static_cast<const __bf16*>(q);
  if (G <= 64) {
    const int chunk = std::min(8, 64 / G);
    for (int r0 = 0; r0 < n; r0 += chunk) {
      const size_t heads = (size_t)r0 * Hq;
      const hipError_t e = launch_partials_tiles(
          Q + heads * HD, kc, vc, pos, part_o + heads * NS * HD, part_ml + heads * NS * 2,
          std::min(chunk, n - r0), Hq, Hkv, max_len, NS, scale, stream, kv8, k_scale, r0);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  const int SG = (G + 63) / 64;                     // sub-groups per KV head
  const size_t kv_head = (size_t)max_len * HD * (kv8 ? 1 : 2);  // cache bytes per KV head
  for (int t = 0; t < n; ++t)
    for (int g = 0; g < Hkv; ++g)
      for (int u = 0; u < SG; ++u) {
        const int h0 = g * G + u * G / SG, h1 = g * G + (u + 1) * G / SG;
        const size_t head = (size_t)t * Hq + h0;
        const hipError_t e = launch_partials_tiles(
            Q + head * HD, static_cast<const char*>(kc) + g * kv_head,
            static_cast<const char*>(vc) + g * kv_head, pos, part_o + head * NS * HD,
            part_ml + head * NS * 2, 1, h1 - h0, 1, max_len, NS, scale, stream, kv8, k_scale, t);
        if (e != hipSuccess) return e;
      }
  return hipSuccess;
}

}  // namespace qe

using namespace qe;

extern "C" int qe_attn_split_size(int L, int NS) {
  if (L < 1 || NS < 1 || L >= SPLIT_L_MAX) return 0;
  return split_size(L, ns_div(NS));  // the kernels' own arithmetic
}

extern "C" hipError_t qe_attn_decode_partials(const void* q, const void* kc, const void* vc,
                                              const int* pos, float* part_o, float* part_ml,
                                              int n, int Hq, int Hkv, int max_len, int NS,
                                              float scale, hipStream_t stream) {
  hipError_t e = check_decode_shape(n, Hq, Hkv, max_len, NS);
  if (e != hipSuccess) return e;
  if (!aligned16(q) || !aligned16(kc) || !aligned16(vc) || !aligned16(part_o) || !pos || !part_ml)
    return hipErrorInvalidValue;
  return launch_partials(q, kc, vc, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, scale, stream);
}

extern "C" hipError_t qe_attn_decode_combine(const float* part_o, const float* part_ml,
                                             const int* pos, const void* qg, long ldp, void* out,
                                             long ldo, int n, int Hq, int max_len, int NS,
                                             hipStream_t stream) {
  if (n < 1 || n > MAX_DECODE_ROWS || Hq < 1 || NS < 1 || max_len < 1 || !part_o || !part_ml ||
      !pos || !qg || !out)
    return hipErrorInvalidValue;
  return launch_combine(part_o, part_ml, pos, qg, ldp, out, ldo, n, Hq, max_len, NS, stream);
}

extern "C" hipError_t qe_attn_decode(const void* q, const void* kc, const void* vc, const int* pos,
                                     const void* qg, long ldp, float* part_o, float* part_ml,
                                     void* out, long ldo, int n, int Hq, int Hkv, int max_len,
                                     int NS, float scale, hipStream_t stream) {
  hipError_t e = qe_attn_decode_partials(q, kc, vc, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS,
                                         scale, stream);
  if (e != hipSuccess) return e;
  return qe_attn_decode_combine(part_o, part_ml, pos, qg, ldp, out, ldo, n, Hq, max_len, NS,
                                stream);
}

// ---------------------------------------------------------------- decode without caller scratch
// The split-KV partials of qe_attn_decode_noalloc live in this file-scope device array: part_o
// [n][Hq][NS][256] then part_ml [n][Hq][NS][2] (fp32), for at most QE_NOALLOC_MAX_SLOTS (row,
// head, slice) triples. Every GPU the library runs on holds its own copy until the process ends.
// In host code `scratch` names a host-side stand-in, never the device memory: its per-device
// address comes from hipGetSymbolAddress and is used everywhere instead.
static __device__ __align__(256) float scratch[QE_NOALLOC_MAX_SLOTS * (HD + 2)];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_ptr[kMaxDevices] = {};

// The current device's address of `scratch`, looked up once per device (with that device
// current) and kept.
hipError_t scratch_of_current_device(float** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[dev] = static_cast<float*>(p);
  }
  *out = g_scratch_ptr[dev];
  return hipSuccess;
}
}  // namespace

extern "C" hipError_t qe_attn_decode_noalloc(const void* q, const void* kc, const void* vc,
                                             const int* pos, const void* qg, long ldp, void* out,
                                             long ldo, int n, int Hq, int Hkv, int max_len, int NS,
                                             float scale, hipStream_t stream) {
  hipError_t e = check_decode_shape(n, Hq, Hkv, max_len, NS);
  if (e != hipSuccess) return e;
  if ((long long)n * Hq * NS > QE_NOALLOC_MAX_SLOTS) return hipErrorInvalidValue;
  float* base = nullptr;
  e = scratch_of_current_device(&base);
  if (e != hipSuccess) return e;
  float* part_o = base;
  float* part_ml = base + (size_t)QE_NOALLOC_MAX_SLOTS * HD;
  return qe_attn_decode(q, kc, vc, pos, qg, ldp, part_o, part_ml, out, ldo, n, Hq, Hkv, max_len,
                        NS, scale, stream);
}

static bool kv_scales_ok(float k_scale, float v_scale) {
  return kv_scale_ok(k_scale) && kv_scale_ok(v_scale);
}

extern "C" hipError_t qe_attn_decode_fp8_partials(const void* q, const void* kc8, const void* vc8,
                                                  const int* pos, float* part_o, float* part_ml,
                                                  int n, int Hq, int Hkv, int max_len, int NS,
                                                  float scale, float k_scale,
                                                  hipStream_t stream) {
  hipError_t e = check_decode_shape(n, Hq, Hkv, max_len, NS);
  if (e != hipSuccess) return e;
  if (!kv_scales_ok(k_scale, 1.f)) return hipErrorInvalidValue;
  if (!aligned16(q) || !aligned16(kc8) || !aligned16(vc8) || !aligned16(part_o) || !pos ||
      !part_ml)
    return hipErrorInvalidValue;
  return launch_partials(q, kc8, vc8, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, scale,
                         stream, true, k_scale);
}

extern "C" hipError_t qe_attn_decode_fp8(const void* q, const void* kc8, const void* vc8,
                                         const int* pos, const void* qg, long ldp, float* part_o,
                                         float* part_ml, void* out, long ldo, int n, int Hq,
                                         int Hkv, int max_len, int NS, float scale, float k_scale,
                                         float v_scale, hipStream_t stream) {
  if (!kv_scales_ok(k_scale, v_scale) || !qg || !out) return hipErrorInvalidValue;
  hipError_t e = qe_attn_decode_fp8_partials(q, kc8, vc8, pos, part_o, part_ml, n, Hq, Hkv,
                                             max_len, NS, scale, k_scale, stream);
  if (e != hipSuccess) return e;
  return launch_combine(part_o, part_ml, pos, qg, ldp, out, ldo, n, Hq, max_len, NS, stream,
                        v_scale);
}

extern "C" hipError_t qe_attn_prep(const void* qg, const void* k, const void* v, long ldp,
                                   const void* qnw, const void* knw, const float* inv_freq,
                                   const int* pos, void* q_out, void* kc, void* vc, int n, int Hq,
                                   int Hkv, int max_len, int rd, float eps, hipStream_t stream);

extern "C" hipError_t qe_attn_prep_decode(const void* qg, const void* k, const void* v, long ldp,
                                          const void* qnw, const void* knw, const float* inv_freq,
                                          const int* pos, void* q_out, void* kc, void* vc,
                                          float* part_o, float* part_ml, void* out, long ldo,
                                          int n, int Hq, int Hkv, int max_len, int rd, int NS,
                                          float scale, float eps, hipStream_t stream) {
  hipError_t e = check_decode_shape(n, Hq, Hkv, max_len, NS);
  if (e != hipSuccess) return e;
  if (rd < 0 || rd > HD || (rd & 1) || ldp < 1 || !qg || !k || !v || !qnw || !knw ||
      !inv_freq || !pos || !q_out || !kc || !vc || !part_o || !part_ml || !out)
    return hipErrorInvalidValue;
  if (!aligned16(q_out) || !aligned16(kc) || !aligned16(vc) || !aligned16(part_o))
    return hipErrorInvalidValue;
  const int NT = ((Hq / Hkv) * n + 15) / 16;
  // Shapes wider than one column tile, rotary parts with more table entries than threads or not
  // a multiple of 8 dims, and input rows the 16-byte loads cannot read: the prep kernel, then the
  // decode. (Two column tiles fused, 3-5 rows at GQA 6, measured slower than the two ops: 25.9
  // against 18.9 us per layer-call at 5 rows on a 4k cache, same bits.)
  if (NT > 1 || n > 8 || rd == 0 || rd % 8 != 0 || n * (rd / 2) > ROPE_TAB || ldp % 8 != 0 ||
      !aligned16(qg) || !aligned16(k) || !aligned16(qnw) || !aligned16(knw) ||
      !aligned16(inv_freq)) {
    e = qe_attn_prep(qg, k, v, ldp, qnw, knw, inv_freq, pos, q_out, kc, vc, n, Hq, Hkv, max_len,
                     rd, eps, stream);
    if (e != hipSuccess) return e;
    return qe_attn_decode(q_out, kc, vc, pos, qg, ldp, part_o, part_ml, out, ldo, n, Hq, Hkv,
                          max_len, NS, scale, stream);
  }
  const dim3 grid(max_slices(max_len, NS), Hkv);
  const NsDiv nd = ns_div(NS);
  const PrepIn pin{static_cast<const __bf16*>(qg), static_cast<const __bf16*>(k),
                   static_cast<const __bf16*>(v), ldp, static_cast<const __bf16*>(qnw),
                   static_cast<const __bf16*>(knw), inv_freq, static_cast<__bf16*>(q_out), rd,
                   eps};
  const float scale_log2 = scale * 1.4426950408889634f;
  const auto* K = static_cast<const __bf16*>(kc);
  const auto* V = static_cast<const __bf16*>(vc);
  if (n == 1)
    attn_partials_kernel<1, true, false><<<grid, dim3(waves_for<1>() * WAVE), 0, stream>>>(
        nullptr, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, pin, 0);
  else
    attn_partials_kernel<1, true><<<grid, dim3(waves_for<1>() * WAVE), 0, stream>>>(
        nullptr, K, V, pos, part_o, part_ml, n, Hq, Hkv, max_len, NS, nd, scale_log2, pin, 0);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  return qe_attn_decode_combine(part_o, part_ml, pos, qg, ldp, out, ldo, n, Hq, max_len, NS,
                                stream);
}

// ---------------------------------------------------------------------------- measurement only
namespace qe {
// The K and V bytes a 1-row decode call reads, with the partials kernel's grid, its slicing (from
// the device scalar pos, as the decode does) and no arithmetic: workgroup (s, g) streams rows
// [s*CH, min((s+1)*CH, L)) of K and V of KV head g, 256 threads, 8 + 8 sixteen-byte
// non-temporal loads in flight per thread. Its time bounds any kernel that must read those bytes
// with that grid.
__global__ void __launch_bounds__(256)
kv_stream_probe_kernel(const __bf16* __restrict__ kc, const __bf16* __restrict__ vc,
                       const int* __restrict__ pos_ptr, int max_len, NsDiv nd,
                       uint32_t* __restrict__ sink) {
  const int L = min(pos_ptr[0] + 1, max_len);
  const int CH = split_size(L, nd);
  const int s = blockIdx.x, g = blockIdx.y;
  const int beg = s * CH, end = min(beg + CH, L);
  if (beg >= end) return;
  const size_t head = (size_t)g * max_len * HD;
  const uint32_t bytes = (uint32_t)end * (HD * 2);
  const __amdgpu_buffer_rsrc_t kr = make_rsrc_uniform(kc + head, bytes);
  const __amdgpu_buffer_rsrc_t vr = make_rsrc_uniform(vc + head, bytes);
  uint32_t acc = 0;
  // rounds of 32 KB per array from the slice start: the round count bounds the loop (an offset
  // stepped past 2^32 would wrap)
  const uint32_t rounds = ((uint32_t)(end - beg) * (HD * 2) + 32767u) / 32768u;
  for (uint32_t r = 0, off = (uint32_t)beg * (HD * 2) + threadIdx.x * 16; r < rounds;
       ++r, off += 256 * 16 * 8) {
    u32x4_t a[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      a[j] = buffer_load16_stream(kr, off + j * 4096);  // past the slice end: 0, no traffic
      b[j] = buffer_load16_stream(vr, off + j * 4096);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      acc ^= a[j][0] ^ a[j][1] ^ a[j][2] ^ a[j][3] ^ b[j][0] ^ b[j][1] ^ b[j][2] ^ b[j][3];
  }
  if (acc == 0x9E3779B9u) sink[0] = acc;
}

// The same K and V bytes (L = min(pos+1, max_len) positions per KV head) on any grid: workgroup
// (s, g) of (GH, Hkv) streams a 4 KB-aligned 1/GH share of KV head g's K rows and of its V rows,
// 256 threads, DEPTH + DEPTH sixteen-byte non-temporal loads in flight per thread (one round),
// no arithmetic. Swept over GH and DEPTH, its fastest time is the floor of reading these bytes in
// one launch on this part, whatever the grid.
template <int DEPTH>
__global__ void __launch_bounds__(256)
kv_stream_sweep_kernel(const char* __restrict__ kc, const char* __restrict__ vc,
                       const int* __restrict__ pos_ptr, int max_len, uint32_t* __restrict__ sink) {
  const int L = min(pos_ptr[0] + 1, max_len);
  const int s = blockIdx.x, g = blockIdx.y, GH = gridDim.x;
  const uint64_t hb = (uint64_t)L * (HD * 2);  // < 2^32 - 32 KB (host check)
  const uint64_t chunk = ((hb + GH - 1) / GH + 4095u) & ~4095ull;
  if ((uint64_t)s * chunk >= hb) return;
  const uint32_t beg = (uint32_t)(s * chunk);
  const uint32_t end = (uint32_t)min((uint64_t)beg + chunk, hb);
  const size_t head = (size_t)g * max_len * (HD * 2);
  const __amdgpu_buffer_rsrc_t kr = make_rsrc_uniform(kc + head, end);
  const __amdgpu_buffer_rsrc_t vr = make_rsrc_uniform(vc + head, end);
  const uint32_t rounds = (end - beg + 4096u * DEPTH - 1) / (4096u * DEPTH);
  uint32_t acc = 0;
  for (uint32_t r = 0, off = beg + threadIdx.x * 16; r < rounds; ++r, off += 4096u * DEPTH) {
    u32x4_t a[DEPTH], b[DEPTH];
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) {
      a[j] = buffer_load16_stream(kr, off + j * 4096);  // past the share's end: 0, no traffic
      b[j] = buffer_load16_stream(vr, off + j * 4096);
    }
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) acc ^= a[j][0] ^ a[j][3] ^ b[j][0] ^ b[j][3];
  }
  if (acc == 0x9E3779B9u) sink[0] = acc;
}

__global__ void __launch_bounds__(WAVE) launch_probe_kernel() {}
}  // namespace qe

extern "C" hipError_t qe_kv_stream_probe(const void* kc, const void* vc, const int* pos, int Hkv,
                                         int max_len, int NS, void* sink, hipStream_t stream) {
  if (max_len < 1 || Hkv < 1 || NS < 1 || !kc || !vc || !pos || !sink ||
      (unsigned long long)(max_len + 64) * HD * 2 >= (1ull << 32))
    return hipErrorInvalidValue;
  kv_stream_probe_kernel<<<dim3(max_slices(max_len, NS), Hkv), dim3(256), 0, stream>>>(
      static_cast<const __bf16*>(kc), static_cast<const __bf16*>(vc), pos, max_len, ns_div(NS),
      static_cast<uint32_t*>(sink));
  return hipGetLastError();
}

extern "C" hipError_t qe_kv_stream_sweep(const void* kc, const void* vc, const int* pos, int Hkv,
                                         int max_len, int grid_per_head, int depth, void* sink,
                                         hipStream_t stream) {
  if (max_len < 1 || Hkv < 1 || grid_per_head < 1 || grid_per_head > 65535 || !kc || !vc ||
      !pos || !sink || (unsigned long long)(max_len + 64) * HD * 2 >= (1ull << 32))
    return hipErrorInvalidValue;
  const dim3 grid(grid_per_head, Hkv);
  const auto* K = static_cast<const char*>(kc);
  const auto* V = static_cast<const char*>(vc);
  auto* S = static_cast<uint32_t*>(sink);
  switch (depth) {
    case 4: kv_stream_sweep_kernel<4><<<grid, dim3(256), 0, stream>>>(K, V, pos, max_len, S); break;
    case 8: kv_stream_sweep_kernel<8><<<grid, dim3(256), 0, stream>>>(K, V, pos, max_len, S); break;
    case 16: kv_stream_sweep_kernel<16><<<grid, dim3(256), 0, stream>>>(K, V, pos, max_len, S); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

extern "C" hipError_t qe_launch_probe(hipStream_t stream) {
  launch_probe_kernel<<<dim3(1), dim3(WAVE), 0, stream>>>();
  return hipGetLastError();
}

extern "C" const char* qe_attn_version(void) { return "qengine_amd attn 0.2 (gfx950)"; }
extern "C" void qe_set_pdl_trigger(int) {}
extern "C" void qe_set_pdl_launch(int) {}
