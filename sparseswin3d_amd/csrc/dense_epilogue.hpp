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
__device__ __forceinline__ void gelu_and_slope(float u, float& g, float& d) {
    const float cdf = 0.5f * (1.f + erff(u * 0.70710678118654752f));
    g = u * cdf;
    d = cdf + u * 0.3989422804014327f * __expf(-0.5f * u * u);
}

// one value: what follows the product, with its column's bias already added
template <int EPI>
__device__ __forceinline__ float finish1(float v, float extra, float& slope) {
    if constexpr (EPI == EPI_RESIDUAL) return v + extra;
    if constexpr (EPI == EPI_SCALE) return v * extra;
    if constexpr (EPI == EPI_GELU) {
        float g;
        gelu_and_slope(v, g, slope);
        return g;
    }
    return v;
}

template <typename T> struct alignas(sizeof(T) * 4) Vec4 { T v[4]; };

struct Epilogue {
    const void* bias;       // [P] of the weights' type, or null
    const void* extra;      // residual [N, P] (type of y) or factor [N, P] (type of the tokens)
    void* y;                // [N, P]
    void* slope;            // GELU: its derivative [N, P] (type of y), or null
};

template <typename T, typename TB, typename TO, int EPI>
__device__ __forceinline__ void finish4(const Epilogue& ep, int64_t row, int col, int P, const f32x4& acc) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = acc[e];
    if (ep.bias) {
        const Vec4<TB> b = *reinterpret_cast<const Vec4<TB>*>(static_cast<const TB*>(ep.bias) + col);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += to_acc(b.v[e]);
    }
    const int64_t at = row * P + col;
    Vec4<TO> s;
    float extra[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (EPI == EPI_RESIDUAL || EPI == EPI_SCALE) {
        using TE = typename std::conditional<EPI == EPI_SCALE, T, TO>::type;
        const Vec4<TE> r = *reinterpret_cast<const Vec4<TE>*>(static_cast<const TE*>(ep.extra) + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) extra[e] = to_acc(r.v[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float d = 0.f;
        v[e] = finish1<EPI>(v[e], extra[e], d);
        s.v[e] = from_acc<TO>(d);
    }
    if constexpr (EPI == EPI_GELU)
        if (ep.slope) *reinterpret_cast<Vec4<TO>*>(static_cast<TO*>(ep.slope) + at) = s;
    Vec4<TO> o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o.v[e] = from_acc<TO>(v[e]);
    *reinterpret_cast<Vec4<TO>*>(static_cast<TO*>(ep.y) + at) = o;
}

// fp32 layers of 96 reduction channels and a multiple of 96 outputs (tall_linear.hip): x [N >= 32, 96], all of Wop in LDS
int staged_layer_96(const float* x, int64_t N, const float* w, int P, bool transposed, int epilogue, const Epilogue& ep, hipStream_t s);

}  // namespace dense
}  // namespace sswin
