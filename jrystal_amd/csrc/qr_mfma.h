// FP64 matrix instruction of gfx950.
#pragma once
#include "common.h"

namespace jrx {

// ------------------------------------------------------------- FP64 MFMA --
// v_mfma_f64_16x16x4f64 on one wave: D(16x16) += A(16x4) B(4x16), lane l
// supplies A[l%16][l/16] and B[l/16][l%16]; accumulator register r of lane
// l holds D[4r + l/16][l%16].  Complex products are four real products.
typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4 mfma4(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ d4 d4zero() { return d4{0.0, 0.0, 0.0, 0.0}; }

// Orders a wave's own LDS accesses (stores of some lanes before loads of
// others); no block barrier.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

}  // namespace jrx
