// Operands of 16 x 16 tiles shared by the flash attention kernels (gfx950, wave64).
#pragma once

#include "sswin_common.hpp"

namespace sswin {
namespace flash {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr float LOG2E = 1.4426950408889634f;
constexpr float MASKED = -100.f * LOG2E;       // what sp_add_mask adds, in units of log 2
constexpr int MAX_ROWS = 4096;
constexpr int64_t MAX_TOKENS = 1 << 24;    // row numbers are multiplied in 24 bits

// four reduction slots of one operand row
template <typename T> struct Frag;
template <> struct Frag<float> {
    f32x4 v;
    __device__ __forceinline__ void load(const float* p) { v = *reinterpret_cast<const f32x4*>(p); }
};
template <> struct Frag<__half> {
    f16x4 v;
    __device__ __forceinline__ void load(const __half* p) { v = *reinterpret_cast<const f16x4*>(p); }
};
template <> struct Frag<__hip_bfloat16> {
    s16x4 v;
    __device__ __forceinline__ void load(const __hip_bfloat16* p) { v = *reinterpret_cast<const s16x4*>(p); }
};

__device__ __forceinline__ f32x4 mma(const Frag<float>& a, const Frag<float>& b, f32x4 c) {
#pragma unroll
    for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[s], b.v[s], c, 0, 0, 0);
    return c;
}
__device__ __forceinline__ f32x4 mma(const Frag<__half>& a, const Frag<__half>& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a.v, b.v, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma(const Frag<__hip_bfloat16>& a, const Frag<__hip_bfloat16>& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.v, b.v, c, 0, 0, 0);
}

template <typename T> __device__ __forceinline__ Frag<T> packed(const f32x4& c);
template <> __device__ __forceinline__ Frag<float> packed<float>(const f32x4& c) { return Frag<float>{c}; }
template <> __device__ __forceinline__ Frag<__half> packed<__half>(const f32x4& c) {
    return Frag<__half>{f16x4{(_Float16)c[0], (_Float16)c[1], (_Float16)c[2], (_Float16)c[3]}};
}
template <> __device__ __forceinline__ Frag<__hip_bfloat16> packed<__hip_bfloat16>(const f32x4& c) {
    struct { uint32_t a, b; } w = {pack_bf16(c[0], c[1]), pack_bf16(c[2], c[3])};
    return Frag<__hip_bfloat16>{__builtin_bit_cast(s16x4, w)};
}

template <typename T> __device__ __forceinline__ void store4(T* p, const f32x4& v);
template <> __device__ __forceinline__ void store4<float>(float* p, const f32x4& v) { *reinterpret_cast<f32x4*>(p) = v; }
template <> __device__ __forceinline__ void store4<__half>(__half* p, const f32x4& v) { *reinterpret_cast<f16x4*>(p) = packed<__half>(v).v; }
template <> __device__ __forceinline__ void store4<__hip_bfloat16>(__hip_bfloat16* p, const f32x4& v) {
    *reinterpret_cast<s16x4*>(p) = packed<__hip_bfloat16>(v).v;
}

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(4)));

}  // namespace flash
}  // namespace sswin
