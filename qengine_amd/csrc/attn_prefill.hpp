// The prefill kernels of attn_prefill_wide.hip, launched from attn_prefill.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace qe {

// Whether the column and workgroup counts of a call fit 32 bits.
bool prefill_wide_valid(int T, int Hq, int Hkv);
// Estimated time of a call whose chunk ends the cache, in steps: the time of one tile of 32 positions
// in a full round of units (0.9 us on the bf16 cache, 1.0 us on the fp8 cache). ws: with a workspace.
float prefill_wide_steps(int T, int Hq, int Hkv, int max_len, bool ws);
// Workspace with which a call cuts units into slices; 0 where it never would. At most
// prefill_wide_ws_most(): two slots for every workgroup that runs at once.
size_t prefill_wide_ws_bytes(int T, int Hq, int Hkv, int max_len);
size_t prefill_wide_ws_most(int Hkv);
// ws: prefill_wide_ws_bytes() bytes, 16-byte aligned, or null (no slices). v_scale multiplies O / l
// before its bf16 rounding (exactly 1 for the bf16 cache).
hipError_t launch_prefill_wide(const void* q, const void* kc, const void* vc, const int* pos,
                               const void* qg, long ldp, void* out, long ldo, int T, int Hq, int Hkv,
                               int max_len, float scale, bool kv8, float v_scale, float* ws,
                               hipStream_t stream);

}  // namespace qe
