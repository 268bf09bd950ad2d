// Three-way bf16 parts of fp32 values: the cut, the part products that reach fp32 precision, and an
// LDS-only workgroup barrier. See split_kernel.hpp for their error.
#pragma once

#include "gemm_kernel.hpp"

namespace mfr::gemm {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

// Two floats rounded to nearest bf16 and packed, the first in the low half.
__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
    const floatx2 v = {x, y};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// Cuts eight elements: x = p0 + p1 + p2 exactly (p0 the nearest bf16 of x, p1 of x - p0, p2 the
// rest, 8 bits at most) for |x| from 2^-100 to the largest bf16. squares: the running sum of the
// squares of the p0.
__device__ __forceinline__ void cut_eight(const float (&reg)[8], uint32_t (&part)[3][4],
                                          float& squares) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float x = reg[2 * e], y = reg[2 * e + 1];
        part[0][e] = pack_bf16(x, y);
        const bf16x2 pair = __builtin_bit_cast(bf16x2, part[0][e]);
        squares = __builtin_amdgcn_fdot2_f32_bf16(pair, pair, squares, false);
        x -= __uint_as_float(part[0][e] << 16);
        y -= __uint_as_float(part[0][e] & 0xffff0000u);
        part[1][e] = pack_bf16(x, y);
        x -= __uint_as_float(part[1][e] << 16);
        y -= __uint_as_float(part[1][e] & 0xffff0000u);
        part[2][e] = pack_bf16(x, y);
    }
}

// A workgroup barrier that waits for this wavefront's LDS accesses only: global loads in flight
// stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The six part products of fp32 precision, smallest first. The tiles through LDS add them in this
// order, 16-deep step by step, so they give the same bits; the register forms' wavefronts each add
// every eighth step and their sums are added at the end.
constexpr int kPartA[6] = {2, 0, 1, 1, 0, 0};
constexpr int kPartB[6] = {0, 2, 1, 0, 1, 0};

} // namespace mfr::gemm
