// Shared pieces of the prompt-attention kernels (forward and backward): 16-bit MFMA
// operands, packing, and wave-uniform loads.
//
// MFMA 16x16x32 layouts (lane l): A[row = l % 16][k = 8 (l / 16) + i],
// B[k = 8 (l / 16) + i][col = l % 16], D[row = 4 (l / 16) + j][col = l % 16].
#pragma once

#include "kvfp8_common.h"

namespace kvfp8 {

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

template <bool kF16>
__device__ __forceinline__ f32x4_t mma16(u32x4_t a, u32x4_t b, f32x4_t c) {
    if constexpr (kF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b),
                                                     c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                      __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Two floats -> one dword of two 16-bit values, rounded to nearest even (one
// v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32).
template <bool kF16>
__device__ __forceinline__ uint32_t pack2(float x0, float x1) {
    const f32x2_t v = {x0, x1};
    if constexpr (kF16) return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
    else return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// Wave-uniform loads through the scalar data cache: a pointer into the constant
// address space (read-only for the kernel's lifetime) lets the compiler use
// s_load. A plain load of this memory would be a vector load here (the kernel also
// stores to global memory), and the compiler would then wait for every
// vector-memory operation in flight, K/V prefetches included.
typedef __attribute__((address_space(4))) const int64_t* const_i64_ptr;
typedef __attribute__((address_space(4))) const int32_t* const_i32_ptr;

// Bounds [s0, s1) of sequence b, clipped to the packed tokens.
__device__ __forceinline__ void seq_bounds(const void* cu, bool cu64, int b, int64_t total, int64_t* s0, int64_t* s1) {
    int64_t lo, hi;
    if (cu64) {
        const const_i64_ptr p = (const_i64_ptr)cu;
        lo = p[b];
        hi = p[b + 1];
    } else {
        const const_i32_ptr p = (const_i32_ptr)cu;
        lo = p[b];
        hi = p[b + 1];
    }
    *s0 = lo < 0 ? 0 : lo;
    *s1 = hi > total ? total : hi;
}

}  // namespace

}  // namespace kvfp8
