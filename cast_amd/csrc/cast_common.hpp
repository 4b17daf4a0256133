// Shared device helpers for the gfx950 tree-verification kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/cast_amd.h"

namespace cast {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kMaxPack = 128;      // two 64-bit ancestor words per row
constexpr int kWave = 64;

__device__ __forceinline__ float bf16_to_float(uint16_t h) {
    return __builtin_bit_cast(float, (uint32_t)h << 16);
}

// Round-to-nearest-even float -> bf16 pair (v_cvt_pk_bf16_f32 on gfx950).
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    bf16x2 p = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, p);
}

// Round-to-nearest-even float -> IEEE half pair (v_cvt_pk_f16_f32 on gfx950).
__device__ __forceinline__ uint32_t pack_f16x2(float lo, float hi) {
    f16x2 p = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, p);
}

__device__ __forceinline__ float f16_to_float(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

// The two 16-bit element formats of the MFMA attention kernels: the 8-wide
// operand of v_mfma_f32_32x32x16_{bf16,f16}, that product, the rounding of
// a float pair to the format and the widening of one element.
struct Bf16 {
    using vec8 = bf16x8;
    static __device__ __forceinline__ floatx16 mma(vec8 a, vec8 b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) { return pack_bf16x2(lo, hi); }
    static __device__ __forceinline__ float widen(uint16_t h) { return bf16_to_float(h); }
    // a float pair as the sum of kTerms pairs of the format, the largest
    // first: three truncations of 8 bits each hold all 24 bits
    static constexpr int kTerms = 3;
    static constexpr float kTermShift = 0.f, kTermSlack = 8.f;
    static __device__ __forceinline__ void split2(float lo, float hi, uint32_t (&w)[3]) {
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const uint32_t bl = __builtin_bit_cast(uint32_t, lo), bh = __builtin_bit_cast(uint32_t, hi);
            w[t] = __builtin_amdgcn_perm(bh, bl, 0x07060302u);
            lo -= __builtin_bit_cast(float, bl & 0xffff0000u);
            hi -= __builtin_bit_cast(float, bh & 0xffff0000u);
        }
    }
};
// A float pair as the sum of three bf16 pairs, each the rounding of what the
// ones before it leave: 8 bits a term and signed remainders hold all 24 bits
// (of values that do not round to infinity).
__device__ __forceinline__ void split_bf16x3(float lo, float hi, uint32_t &w0, uint32_t &w1, uint32_t &w2) {
    w0 = pack_bf16x2(lo, hi);
    lo -= __builtin_bit_cast(float, w0 << 16);
    hi -= __builtin_bit_cast(float, w0 & 0xffff0000u);
    w1 = pack_bf16x2(lo, hi);
    lo -= __builtin_bit_cast(float, w1 << 16);
    hi -= __builtin_bit_cast(float, w1 & 0xffff0000u);
    // (what is left has at most 8 bits: the upper half is all of it)
    w2 = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302u);
}

struct Fp16 {
    using vec8 = f16x8;
    static __device__ __forceinline__ floatx16 mma(vec8 a, vec8 b, floatx16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) { return pack_f16x2(lo, hi); }
    static __device__ __forceinline__ float widen(uint16_t h) { return f16_to_float(h); }
    // Two roundings of 11 bits each leave 2^-24 of the value, as float does,
    // while the second term is a normal half: values of up to 1 are scaled by
    // 2^kTermShift, the most that fits (with no slack, kTermSlack, above 1).
    // Down to 2^-16 that is so; below, 2^-40 is what is left.
    static constexpr int kTerms = 2;
    static constexpr float kTermShift = 15.f, kTermSlack = 0.f;
    static __device__ __forceinline__ void split2(float lo, float hi, uint32_t (&w)[2]) {
        w[0] = pack_f16x2(lo, hi);
        w[1] = pack_f16x2(lo - f16_to_float((uint16_t)w[0]), hi - f16_to_float((uint16_t)(w[0] >> 16)));
    }
};

__device__ __forceinline__ void raise_flag(int32_t *status, int32_t bit) {
    if (status) atomicOr(status, bit);
}

// The value held by lane (l ^ 32).
__device__ __forceinline__ float partner32(float x) { return __shfl_xor(x, 32); }

}  // namespace cast
