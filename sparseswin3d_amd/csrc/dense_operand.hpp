// Operands of the matrix instructions of the dense layers (dense.hip, dense_pairs.hip, mlp.hip): fp32 values as three bf16 pieces or two
// fp16 pieces, 16-bit values as they are, and the copies from memory to LDS that pass no register.
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

// fp32 values as two fp16 pieces, h rounded to nearest and l, 2^11 times what is left of it, also rounded: x 2^e = h + l 2^-11 to 2^-23 of
// the power of two above x, so three products of 11 bits each take the place of six of 8: (h,h), and (l,h) (h,l) into sums of their own, for
// their factor (published as error-corrected half-precision products: Ootomo and Yokota, "Recovering single precision accuracy from Tensor
// Cores while surpassing the FP32 theoretical peak performance", 2022; here with a scale per row and column).
// Half the matrix instructions, two thirds of the operand bytes and half the vector instructions.  What is lost: a bit of a
// quarter of the values (6e-8 of a result, with l l); what is won: the matrix instructions do not round their sums to nearest, and
// (h,h) is one of them a step, in place of six.  Infinities and NaN leave NaN, as above.
// fp16 has five bits of exponent, so rows (and columns) are scaled by a power of two: fixed, so that the largest value lies in [2^14, 2^15), or
// following the largest value so far, which then lies above 2^12 (pairs_rows_kernel, hidden values of mlp_kernel).  Scaled values
// from 2^-13 on keep all bits, since l is of h's size: down to 2^-27 of the row's largest, 2^-25 of the largest so far.  Smaller ones are off by up to
// 2^-36, so a sum of K products, each with a factor below 2^15, by up to K 2^-20.  Sums of at least PAIRS_SMALL are therefore right to K 2^-26 of themselves, a
// quarter of what K roundings of plain fp32 may add up to; smaller ones, unless row or column is all zeros, are formed again in plain fp32
// (normally distributed operands: one in 2^20 and fewer).
struct Pairs {
    static constexpr float LOW = 0.00048828125f;                         // 2^-11
    static __device__ __forceinline__ f32x16 mfma(const u32x4& a, const u32x4& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
    }
};
__device__ __forceinline__ void split_pairs(const float (&v)[8], float scale, u32x4 (&out)[2]) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float a = v[2 * q], b = v[2 * q + 1];
        f16x2 h = {(_Float16)(a * scale), (_Float16)(b * scale)};
        asm("" : "+v"(h));                                               // (or each half is converted again for its rest)
        const f16x2 l = {(_Float16)(fmaf(a, scale, -(float)h[0]) * 2048.f), (_Float16)(fmaf(b, scale, -(float)h[1]) * 2048.f)};
        out[0][q] = __builtin_bit_cast(uint32_t, h);
        out[1][q] = __builtin_bit_cast(uint32_t, l);
    }
}
constexpr float PAIRS_SMALL = 64.f;
// exponent E with |v| < 2^E; of zero far below that of any value.  (Infinities and NaN: 0.)
__device__ __forceinline__ int exponent_above(float most) { return most == 0.f ? -200 : __builtin_amdgcn_frexp_expf(most); }
// Exponent of the scale of a row whose largest value lies below 2^above.  Scales stay normal numbers; exponents above PAIRS_MOST_SCALE
// say that the row (so far) is all zeros; its scale is 2^PAIRS_MOST_SCALE or 0, never infinite, which would turn the zeros into NaN.
constexpr int PAIRS_MOST_SCALE = 120, PAIRS_ZEROS = 121, PAIRS_ZEROS_SO_FAR = 200;
__device__ __forceinline__ int pairs_scale(int above) { return above == -200 ? PAIRS_ZEROS : min(15 - above, PAIRS_MOST_SCALE); }
// The same where it follows the largest value: from e on to a step whose values lie below 2^above (above + e > 15: they would leave fp16's range)
__device__ __forceinline__ int pairs_scale_after(int above, int e) { return above + e > 15 ? min(13 - above, PAIRS_MOST_SCALE) : e; }
__device__ __forceinline__ float power_of_two(int e) { return __builtin_amdgcn_ldexpf(1.f, e); }
__device__ __forceinline__ float largest(const float (&v)[8]) {
    float m = fabsf(v[0]);
#pragma unroll
    for (int e = 1; e < 8; ++e) m = fmaxf(m, fabsf(v[e]));
    return m;
}
// The least value that is not zero, as a number that grows with it (0xffffffff: none so far), and whether pieces of that scale lose bits of it
__device__ __forceinline__ uint32_t least_nonzero(const float (&v)[8], uint32_t m) {
#pragma unroll
    for (int e = 0; e < 8; ++e) m = min(m, (__builtin_bit_cast(uint32_t, v[e]) << 1) - 1u);
    return m;
}
__device__ __forceinline__ bool pairs_lose(uint32_t least, float scale) {
    return least != 0xffffffffu && __builtin_bit_cast(float, (least + 1u) >> 1) * scale < 0x1p-13f;
}
// of a lane and the one 32 lanes away
__device__ __forceinline__ float largest_of_halves(float m) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, m), __builtin_bit_cast(uint32_t, m), false, false);
    return fmaxf(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}

// Pieces of the columns [32 tile, 32 tile + 32) of Wop [K, P] (W [P, K] turned, or with DOWN W [K, P] itself), a scale per column, by a workgroup of
// WAVES wavefronts: put(column, step of 16 channels, half of it, pieces); columns past the last repeat it.  Returns the exponent of the
// scale of the lane's column, to all; with LOST, PAIRS_LOST more where the pieces lose bits.
constexpr int PAIRS_LOST = 1024;
template <bool DOWN, int WAVES, bool LOST, typename PUT>
__device__ __forceinline__ int pairs_of_columns(const float* __restrict__ w, int K, int P, int tile, PUT put) {
    constexpr int KEPT = 4;                                              // steps of a wavefront in registers: 64 WAVES channels are read once
    __shared__ float most[WAVES][32];
    __shared__ uint32_t leasts[LOST ? WAVES : 1][32];
    const int wave = threadIdx.x >> 6, half = (threadIdx.x & 63) >> 5, l32 = threadIdx.x & 31;
    const int col = min(tile * 32 + l32, P - 1), steps = K / 16;
    auto load = [&](int ks, float (&v)[8]) {
        const int k = ks * 16 + half * 8;
        if constexpr (DOWN) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = w[(int64_t)(k + e) * P + col];
        } else {
            const f32x4* src = reinterpret_cast<const f32x4*>(w + (int64_t)col * K + k);
            const f32x4 a = src[0], b = src[1];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = e < 4 ? a[e] : b[e - 4];
        }
    };
    float kept[KEPT][8], m = 0.f;
    uint32_t least = 0xffffffffu;
    auto see = [&](const float (&v)[8]) {
        m = fmaxf(m, largest(v));
        if constexpr (LOST) least = least_nonzero(v, least);
    };
#pragma unroll
    for (int i = 0; i < KEPT; ++i)
        if (wave + i * WAVES < steps) load(wave + i * WAVES, kept[i]);
#pragma unroll
    for (int i = 0; i < KEPT; ++i)
        if (wave + i * WAVES < steps) see(kept[i]);
    for (int ks = wave + KEPT * WAVES; ks < steps; ks += WAVES) {
        float v[8];
        load(ks, v);
        see(v);
    }
    m = largest_of_halves(m);
    if constexpr (LOST) least = min(least, (uint32_t)__shfl_xor((int)least, 32, 64));
    if (half == 0) {
        most[wave][l32] = m;
        if constexpr (LOST) leasts[wave][l32] = least;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < WAVES; ++q) {
        m = fmaxf(m, most[q][l32]);
        if constexpr (LOST) least = min(least, leasts[q][l32]);
    }
    const int e = pairs_scale(exponent_above(m));
    const float scale = power_of_two(e);
    u32x4 p[2];
#pragma unroll
    for (int i = 0; i < KEPT; ++i)
        if (wave + i * WAVES < steps) {
            split_pairs(kept[i], scale, p);
            put(tile * 32 + l32, wave + i * WAVES, half, p);
        }
    for (int ks = wave + KEPT * WAVES; ks < steps; ks += WAVES) {
        float v[8];
        load(ks, v);
        split_pairs(v, scale, p);
        put(tile * 32 + l32, ks, half, p);
    }
    return LOST && pairs_lose(least, scale) ? e + PAIRS_LOST : e;
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

__device__ __forceinline__ float wave_sum(float v) {
    v = row16_sum(v);
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}
// the smaller of |a| and |b|, NaN where one is; whether results of a row whose scale's exponent is e, the least of them as it left the products, are NaN
// or small
__device__ __forceinline__ float least_size(float a, float b) { return __builtin_elementwise_minimum(fabsf(a), fabsf(b)); }
__device__ __forceinline__ float wave_least(float v) {
#pragma unroll
    for (int m = 32; m; m >>= 1) v = least_size(v, __shfl_xor(v, m, 64));
    return v;
}
__device__ __forceinline__ bool nan_or_small(float least, int e) { return e <= PAIRS_MOST_SCALE ? !(least >= PAIRS_SMALL) : least != least; }
// sum over i < n of a[i] b[i b_step], by a wavefront (a, b uniform), to all its lanes
__device__ __forceinline__ float wave_product(const float* a, const float* b, int64_t b_step, int n) {
    float s = 0.f;
#pragma unroll 1
    for (int i = threadIdx.x & 63; i < n; i += 64) s = fmaf(a[i], b[i * b_step], s);
    return wave_sum(s);
}
// again(lane, bit) for every bit set in the lanes' masks, by the wavefront together: a result formed again takes it 2 us, by a lane alone some 20
template <typename F> __device__ __forceinline__ void for_each_small(uint32_t mask, F again) {
    while (const uint64_t lanes = __ballot(mask != 0)) {
        const int owner = __builtin_ctzll(lanes);
        again(owner, __builtin_ctz((uint32_t)__builtin_amdgcn_readlane((int)mask, owner)));
        if ((int)(threadIdx.x & 63) == owner) mask &= mask - 1;
    }
}
// more of them, by lane, than one by one pays for
__device__ __forceinline__ bool many_small(uint32_t mask) { return __popcll(__ballot(mask != 0)) > 8; }

// a last ragged tile is moved back to end at row N, tiles behind it repeat it: rows stored twice hold the same bits
__device__ __forceinline__ int64_t tile_row(int64_t t, int64_t N) { return t * 32 + 32 <= N ? t * 32 : N - 32; }
// workgroups b, b + 8, b + 16 ... share an XCD and its L2: the column blocks of one row block are dealt to such workgroups
__device__ __forceinline__ void block_of(int groups, int& cg, int64_t& rb) {
    const int b = blockIdx.x, chunk = 8 * groups, full = gridDim.x / chunk * chunk;
    if (b < full) {
        cg = (b / 8) % groups;
        rb = b / chunk * 8 + b % 8;
    } else {
        cg = (b - full) % groups;
        rb = full / groups + (b - full) / groups;
    }
}

// 64 lanes x 16 bytes: lane l's piece lands at lds + 16 l
__device__ __forceinline__ void copy_to_lds(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
// 16 bytes a lane, counted by the waits that follow.  The registers of a store this wide may not be written by the next
// instruction, which the compiler sees to for its own stores only.
__device__ __forceinline__ void store_counted(void* p, const u32x4& v) {
    asm volatile("global_store_dwordx4 %0, %1, off\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}
template <int N> __device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ void block_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace dense
}  // namespace sswin
