// 32-bit matrix instructions and what goes with them in the chunked recurrences.
#pragma once
#include "seq_common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// 16 x 16 += 16 x 4 * 4 x 16. Lane l holds a[l % 16][l / 16], b[l / 16][l % 16] and c[4 (l / 16) + 0..3][l % 16].
__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// A barrier for data in LDS only: __syncthreads would also wait for every global load in flight, and the next chunk's loads are
// meant to stay in flight across the barriers of this one.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
