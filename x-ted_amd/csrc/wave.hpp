// Wave64 DPP helpers shared by the forest kernels (gfx950).
#pragma once
#include <hip/hip_runtime.h>

#include <climits>

namespace xted {

constexpr int kBig = INT_MAX / 4;

// DPP control codes (GFX9 encoding).
#define DPP_ROW_SHR(n) (0x110 + (n))
#define DPP_WAVE_SHR1 0x138
#define DPP_ROW_BCAST15 0x142
#define DPP_ROW_BCAST31 0x143

// Inclusive prefix minimum over the 64 lanes of a wave (lane order). A lane
// whose DPP source is out of range (or whose row the mask leaves out) reads
// INT_MAX, the identity of min; with that identity as the "old" operand the
// compiler fuses each move into its min (one v_min_i32 with a DPP source).
__device__ __forceinline__ int wave_incl_min(int v) {
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_SHR(1), 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_SHR(2), 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_SHR(4), 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_SHR(8), 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_BCAST15, 0xa, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(INT_MAX, v, DPP_ROW_BCAST31, 0xc, 0xf, false));
  return v;
}

// Value of lane-1 (lane 0 receives `fill`).
__device__ __forceinline__ int wave_shr1(int v, int fill) {
  return __builtin_amdgcn_update_dpp(fill, v, DPP_WAVE_SHR1, 0xf, 0xf, false);
}

// Words of a TD row group: 2, 4 or 8 entries of 16 bits (td_t), two to a
// 32-bit word, at any even byte address (the target's unaligned-access mode
// lets one dwordx2 / dwordx4 load read them).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// Word 3 of a raw buffer resource on CDNA (32-bit data format, no swizzle).
constexpr int32_t kBufferWord3 = 0x00020000;

}  // namespace xted
