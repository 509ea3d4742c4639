// What follows the product of a dense layer, shared by the kernels of dense.hip and tall_linear.hip.
#pragma once

#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "sswin_common.hpp"

namespace sswin {
namespace dense {

typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { EPI_NONE = SSWIN_DENSE_PLAIN, EPI_GELU = SSWIN_DENSE_GELU, EPI_RESIDUAL = SSWIN_DENSE_RESIDUAL, EPI_SCALE = SSWIN_DENSE_SCALE };

// ------------------------------------------------------------------------------------------
// the last step on four consecutive columns of a row
// ------------------------------------------------------------------------------------------
// u Phi(u) and its derivative.  1 - Phi(|u|) = exp(-u^2/2) Q(t), t = 1/(1 + c|u|) (Hastings' form); for fp32 results and
// |u| < 1 Phi = 1/2 + u R(u^2).  Q and R are least squares fits made for this file (to 1.4e-8 and 3e-10).  fp32: Phi to 9e-8,
// u Phi to 4e-7 up to |u| = 12, as the form with erff; 16 bit (Q alone): 2.3e-7 and 4e-7, a thousandth of their rounding.
// No branch, and the exponential serves both results: with erff the vector units bound the feed-forward layers (219 000 rows
// 96 -> 384 bf16 with the derivative: 171 us, without the step 53).
template <bool WIDE>
__device__ __forceinline__ void gelu_and_slope(float u, float& g, float& d) {
    const float a = fabsf(u), s = u * u, e = __builtin_amdgcn_exp2f(s * -0.72134752044f), t = __builtin_amdgcn_rcpf(fmaf(a, 0.282842726f, 1.f));
    float q = fmaf(-0.100168057f, t, 0.354737073f);
    q = fmaf(fmaf(fmaf(fmaf(q, t, -0.185730487f), t, 0.234369889f), t, 0.080814302f), t, 0.115977287f) * t * e;
    float cdf = u < 0.f ? q : 1.f - q;
    if constexpr (WIDE) {
        float r = fmaf(-7.66468293e-06f, s, 0.000113512666f);
        r = fmaf(fmaf(fmaf(fmaf(r, s, -0.00118635304f), s, 0.00997333135f), s, -0.0664903596f), s, 0.398942292f);
        cdf = a < 1.f ? fmaf(u, r, 0.5f) : cdf;
    }
    g = u * cdf;
    d = fmaf(u * 0.3989422804014327f, e, cdf);
}

// one value: what follows the product, with its column's bias already added
template <int EPI, bool WIDE = true>
__device__ __forceinline__ float finish1(float v, float extra, float& slope) {
    if constexpr (EPI == EPI_RESIDUAL) return v + extra;
    if constexpr (EPI == EPI_SCALE) return v * extra;
    if constexpr (EPI == EPI_GELU) {
        float g;
        gelu_and_slope<WIDE>(v, g, slope);
        return g;
    }
    return v;
}

template <typename T> struct alignas(sizeof(T) * 4) Vec4 { T v[4]; };

template <typename T> __device__ __forceinline__ uint32_t pack2(float a, float b);
template <> __device__ __forceinline__ uint32_t pack2<__half>(float a, float b) {
    return (uint32_t)__half_as_ushort(__float2half(a)) | ((uint32_t)__half_as_ushort(__float2half(b)) << 16);
}
template <> __device__ __forceinline__ uint32_t pack2<__hip_bfloat16>(float a, float b) {
    return pack_bf16(a, b);
}
template <typename T> __device__ __forceinline__ Vec4<T> pack4(const float (&v)[4]) {
    if constexpr (sizeof(T) == 4) {
        return Vec4<T>{v[0], v[1], v[2], v[3]};
    } else {
        struct { uint32_t a, b; } w = {pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
        return __builtin_bit_cast(Vec4<T>, w);
    }
}

struct Epilogue {
    const void* bias;       // [P] of the operands' type, or null
    const void* extra;      // residual [N, P] (type of y) or factor [N, P] (type of the tokens)
    void* y;                // [N, P]
    void* slope;            // GELU: its derivative [N, P] (type of y), or null
};

// residual or factor of four consecutive columns (loaded ahead of the last step, which would wait for it)
template <typename T, typename TO, int EPI> struct Second4 {
    static constexpr bool USED = EPI == EPI_RESIDUAL || EPI == EPI_SCALE;
    using TE = typename std::conditional<EPI == EPI_SCALE, T, TO>::type;
    Vec4<TE> r;
    __device__ __forceinline__ void load(const Epilogue& ep, int64_t row, int col, int P) {
        if constexpr (USED) r = *reinterpret_cast<const Vec4<TE>*>(static_cast<const TE*>(ep.extra) + row * P + col);
    }
};

template <typename T, typename TO, int EPI>
__device__ __forceinline__ void finish4(const Epilogue& ep, int64_t row, int col, int P, const f32x4& acc, const Second4<T, TO, EPI>& second) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = acc[e];
    if (ep.bias) {
        const Vec4<T> b = *reinterpret_cast<const Vec4<T>*>(static_cast<const T*>(ep.bias) + col);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += to_acc(b.v[e]);
    }
    const int64_t at = row * P + col;
    float d[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float extra = 0.f;
        if constexpr (Second4<T, TO, EPI>::USED) extra = to_acc(second.r.v[e]);
        v[e] = finish1<EPI, sizeof(TO) == 4>(v[e], extra, d[e]);
    }
    if constexpr (EPI == EPI_GELU)
        if (ep.slope) *reinterpret_cast<Vec4<TO>*>(static_cast<TO*>(ep.slope) + at) = pack4<TO>(d);
    *reinterpret_cast<Vec4<TO>*>(static_cast<TO*>(ep.y) + at) = pack4<TO>(v);
}

// the same for eight consecutive columns: 16-bit rows are touched in 16-byte pieces
template <typename T> struct alignas(16) Vec8 { Vec4<T> q[2]; };
template <typename T, typename TO, int EPI> struct Second8 {
    using TE = typename Second4<T, TO, EPI>::TE;
    Vec8<TE> r;
    __device__ __forceinline__ void load(const Epilogue& ep, int64_t row, int col, int P) {
        if constexpr (Second4<T, TO, EPI>::USED) r = *reinterpret_cast<const Vec8<TE>*>(static_cast<const TE*>(ep.extra) + row * P + col);
    }
};
template <typename T, typename TO, int EPI>
__device__ __forceinline__ void finish8(const Epilogue& ep, int64_t row, int col, int P, const f32x4 (&acc)[2], const Second8<T, TO, EPI>& second) {
    Vec8<T> b;
    if (ep.bias) b = *reinterpret_cast<const Vec8<T>*>(static_cast<const T*>(ep.bias) + col);
    const int64_t at = row * P + col;
    Vec8<TO> y, slope;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float v[4], d[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float extra = 0.f;
            if constexpr (Second4<T, TO, EPI>::USED) extra = to_acc(second.r.q[h].v[e]);
            v[e] = finish1<EPI, sizeof(TO) == 4>(ep.bias ? acc[h][e] + to_acc(b.q[h].v[e]) : acc[h][e], extra, d[e]);
        }
        y.q[h] = pack4<TO>(v);
        if constexpr (EPI == EPI_GELU) slope.q[h] = pack4<TO>(d);
    }
    if constexpr (EPI == EPI_GELU)
        if (ep.slope) *reinterpret_cast<Vec8<TO>*>(static_cast<TO*>(ep.slope) + at) = slope;
    *reinterpret_cast<Vec8<TO>*>(static_cast<TO*>(ep.y) + at) = y;
}

// fp32 layers of 96 reduction channels and a multiple of 96 outputs with a second operand (tall_linear.hip): x [N >= 32, 96], all of Wop in LDS;
// a residual, or turned a factor
int staged_layer_96(const float* x, int64_t N, const float* w, int P, bool transposed, const Epilogue& ep, hipStream_t s);
// whether a layer of N rows, K -> P, takes the kernel for few rows, whose wavefronts share the reduction (dense.hip)
bool few_rows(int dtype, int64_t N, int K, int P);
// fp32 layers as fp16 pairs (dense_pairs.hip), W's pieces in ws; y and x apart, here and below
inline bool pairs_takes(int K) { return K >= 96; }
size_t pairs_workspace_bytes(int K, int P);
template <int EPI, bool DOWN> int pairs_layer(const float* x, int64_t N, int K, const float* w, int P, const Epilogue& ep, void* ws, hipStream_t s);
// the same for 96 reduction channels and a multiple of 96 outputs, without a workspace; false where staged_layer_96 is ahead (rc untouched)
template <int EPI, bool DOWN> bool pairs_held(const float* x, int64_t N, const float* w, int P, const Epilogue& ep, hipStream_t s, int& rc);
// 16-bit layers of 48, 96 or 192 reduction channels without a last step: x read once (mlp.hip)
bool rows_once_takes(int64_t N, int D, int P);
template <typename T> int rows_once(const T* x, int64_t N, int D, const T* w, const T* b, int P, T* y, hipStream_t s);

}  // namespace dense
}  // namespace sswin
