// Operands of the matrix instructions of the dense layers (dense.hip, mlp.hip): fp32 values as three bf16 pieces, 16-bit values
// as they are, and the copies from memory to LDS that pass no register.
#pragma once

#include <stdint.h>

#include "dense_epilogue.hpp"
#include "mfma_block.hpp"
#include "sswin_common.hpp"

namespace sswin {
namespace dense {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------------------------------
// operand pieces: 8 reduction values of one row as PL planes of 16 bytes
// ------------------------------------------------------------------------------------------
template <typename T> struct Op;
template <> struct Op<float> {
    static constexpr int PL = 3;
    // the six piece products, small terms first: (l,h) (h,l) (m,m) (m,h) (h,m) (h,h)
    static constexpr int NP = 6;
    static constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
    static __device__ __forceinline__ f32x16 mfma(const u32x4& a, const u32x4& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
};
template <> struct Op<__half> {
    static constexpr int PL = 1, NP = 1;
    static constexpr int PA[1] = {0}, PB[1] = {0};
    static __device__ __forceinline__ f32x16 mfma(const u32x4& a, const u32x4& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    }
};
template <> struct Op<__hip_bfloat16> {
    static constexpr int PL = 1, NP = 1;
    static constexpr int PA[1] = {0}, PB[1] = {0};
    static __device__ __forceinline__ f32x16 mfma(const u32x4& a, const u32x4& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
};

// x = h + m + l exactly, h rounded to nearest (a carry of the half into the upper 16 bits), m and l cut off: with x of leading power
// 1, |m| <= 2^-8 and |l| < 2^-16, so that the products left out (m l, l m, l l) stay below 2^-23.  Cutting h off as well, |m| < 2^-7
// and |l| < 2^-15 with x's sign, they reach 2^-21 and add up (equal operands just below 1 + 2^-7: 7.9 x 2^-24 of the result, now
// 2.0 x 2^-24).  The price is two additions a pair: 112 700 rows 48 -> 144 and 48 -> 48 together 48.1 -> 49.1 us, their weight
// gradients 52.2 -> 53.6.  Rounding m as well (2^-24) costs twice that, v_cvt_pk_bf16_f32 in place of the integer forms 20 % of the
// narrow weight gradients, the two missing products 15 % of the wide layers.  From 2^128 - 2^119 on h is infinite: see plain_products.
__device__ __forceinline__ void split2(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
    auto bits = [](float v) { return __builtin_bit_cast(uint32_t, v); };
    auto value = [](uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); };
    auto upper = [](uint32_t hi, uint32_t lo) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); };
    const uint32_t u0 = bits(x0) + 0x8000u, u1 = bits(x1) + 0x8000u;
    const float r0 = x0 - value(u0), r1 = x1 - value(u1);
    h = upper(u1, u0);
    m = upper(bits(r1), bits(r0));
    l = upper(bits(r1 - value(bits(r1))), bits(r0 - value(bits(r0))));
}

// eight fp32 values -> planes of T
template <typename T>
__device__ __forceinline__ void planes_of(const float (&v)[8], u32x4 (&out)[Op<T>::PL]) {
    if constexpr (Op<T>::PL == 3) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint32_t h, m, l;
            split2(v[2 * q], v[2 * q + 1], h, m, l);
            out[0][q] = h, out[1][q] = m, out[2][q] = l;
        }
    } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) out[0][q] = pack2<T>(v[2 * q], v[2 * q + 1]);
    }
}

// Pieces of an infinity hold a NaN, and so does every result one takes part in, as do pieces whose sums leave the range: fp32
// results that come out NaN are formed again from the operands in plain fp32, in the order of the reduction, until they are
// NaN there as well.
__device__ __forceinline__ bool nan_among(const f32x4& v) {
    const float t = (v[0] + v[1]) + (v[2] + v[3]);                       // infinities of both signs too: formed again for nothing
    return t != t;
}
// sum over i < n of a[i a_step] b[i b_step + e b_next], e < 4; four steps of the reduction in flight
__device__ __forceinline__ f32x4 plain_products(const float* a, int64_t a_step, const float* b, int64_t b_step, int64_t b_next, int64_t n) {
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int64_t i0 = 0; i0 < n && (s[0] == s[0] || s[1] == s[1] || s[2] == s[2] || s[3] == s[3]); i0 += 4) {
        float v[4];
        f32x4 w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t i = i0 + q < n ? i0 + q : n - 1;
            v[q] = a[i * a_step];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[q][e] = b[i * b_step + e * b_next];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (i0 + q < n)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = fmaf(v[q], w[q][e], s[e]);
    }
    return s;
}

// 64 lanes x 16 bytes: lane l's piece lands at lds + 16 l
__device__ __forceinline__ void copy_to_lds(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
template <int N> __device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void block_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace dense
}  // namespace sswin
