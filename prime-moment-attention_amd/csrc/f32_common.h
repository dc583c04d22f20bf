// Device helpers shared by the fp32 kernels (chunk_f32.hip, delta_f32.hip and
// delta_bwd.hip): the fp32 MFMA, 16-byte accesses, the lower tiles of a chunk's
// 64 x 64 blocks and the delta chunk's triangular solve.
#pragma once

#include "prefill_common.h"

namespace prime {

// v_mfma_f32_16x16x4_f32: lane l holds A[l%16][k = l/16] and B[k = l/16][l%16];
// the accumulator holds D[4(l/16) + r][l%16]
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 ld4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }
__device__ __forceinline__ f32x4 ld4(const uint8_t *p) { return *reinterpret_cast<const f32x4 *>(p); }
__device__ __forceinline__ void st4(float *p, f32x4 v) { *reinterpret_cast<f32x4 *>(p) = v; }
__device__ __forceinline__ void st4(uint8_t *p, f32x4 v) { *reinterpret_cast<f32x4 *>(p) = v; }

// lower 16x16 tile t (0..9) -> (row block, column block)
__device__ __forceinline__ void lower_tile(int t, int &ib, int &jb) {
    ib = t < 1 ? 0 : t < 3 ? 1 : t < 6 ? 2 : 3;
    jb = t - ib * (ib + 1) / 2;
}

// One column of (I + N)^-1 x in place, N strictly lower with rows of PITCH
// floats: forward substitution in registers, each row's sum in four partial
// sums.  The empty asm statements keep the compiler from hoisting all row
// reads to the top or sinking a row's arithmetic to its last use (either
// spills).
template <int PITCH>
__device__ __forceinline__ void solve_unit_lower(const float *nbase, float (&x)[kC]) {
#pragma unroll
    for (int i = 1; i < kC; ++i) {
        int ro = i * PITCH;
        asm volatile("" : "+v"(ro));
        float acc[4] = {x[i], 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < i; j += 4) {
            const f32x4 n4 = ld4(nbase + ro + j);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (j + e < i) acc[e] -= n4[e] * x[j + e];
        }
        float r = (acc[0] + acc[1]) + (acc[2] + acc[3]);
        asm volatile("" : "+v"(r));
        x[i] = r;
    }
}

}  // namespace prime
