// Row normalisation of a tall [N, D] feature matrix (nn.LayerNorm of sparse_swin/swin3d_base.py:706, 722 and of the
// merge between stages), forward and backward.
//
// Bound by memory: forward x in, y out; backward dy, x (and the gradient that arrives over the residual path) in, dx
// out.  A row is held by L lanes, V pieces of 16 bytes of x per lane (L and V from the row length: the channel counts of
// a stage are 3 * 2^k * 16, so L = D / (3 * 16 bytes) and V = 3 leave no lane idle), so 64 / L rows lie next to each
// other in a wavefront, every access is a run of whole rows, both sums of a row are butterflies over L lanes and
// nothing goes through LDS.  The column sums of the backward (gradients of gain and offset) stay in registers over the
// rows of a wavefront, are added over the workgroup in LDS and over the workgroups by a second kernel, in a fixed order.
// 219 000 rows of 96 fp32 channels: forward 26 us (6.6 TB/s, part of it from the last-level cache), backward with the residual
// gradient 44 us (62 with twice the workgroups and 16 threads per column sum); PyTorch's kernels take 197 us and 299 us (its
// gain / offset sums alone 191).
#include <algorithm>

#include "sswin_common.hpp"

namespace sswin {

template <typename T, int VEC> struct alignas(sizeof(T) * VEC) LnVec { T v[VEC]; };

template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
    if (L >= 2) v += dpp_f32<0xB1>(v);
    if (L >= 4) v += dpp_f32<0x4E>(v);
    if (L >= 8) v += dpp_f32<0x141>(v);
    if (L >= 16) v += dpp_f32<0x140>(v);
    if (L >= 32) v += __shfl_xor(v, 16, 64);
    if (L >= 64) v += __shfl_xor(v, 32, 64);
    return v;
}

constexpr int LN_THREADS = 256;

// EXACT: D == L * V * VEC, otherwise pieces at or beyond D are skipped
template <typename TX, typename TY, typename TP, int L, int V, bool EXACT>
__global__ __launch_bounds__(LN_THREADS) void layer_norm_forward_kernel(const TX* __restrict__ x, int64_t N, int D,
                                                                        const TP* __restrict__ gamma,
                                                                        const TP* __restrict__ beta, float eps,
                                                                        TY* __restrict__ y, float* __restrict__ stats) {
    constexpr int VEC = 16 / sizeof(TX), RPB = LN_THREADS / L;
    const int sub = threadIdx.x % L;
    const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / L;
    if (row >= N) return;
    const TX* xr = x + row * D;
    float v[V][VEC], sum = 0.f;
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int c = (k * L + sub) * VEC;
        if (EXACT || c < D) {
            const LnVec<TX, VEC> p = *reinterpret_cast<const LnVec<TX, VEC>*>(xr + c);
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[k][e] = to_acc(p.v[e]), sum += v[k][e];
        } else {
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[k][e] = 0.f;
        }
    }
    const float inv = 1.f / (float)D, mean = lanes_sum<L>(sum) * inv;
    float sq = 0.f;
#pragma unroll
    for (int k = 0; k < V; ++k)
        if (EXACT || (k * L + sub) * VEC < D)
#pragma unroll
            for (int e = 0; e < VEC; ++e) v[k][e] -= mean, sq += v[k][e] * v[k][e];
    const float rstd = 1.f / sqrtf(lanes_sum<L>(sq) * inv + eps);
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int c = (k * L + sub) * VEC;
        if (EXACT || c < D) {
            const LnVec<TP, VEC> g = *reinterpret_cast<const LnVec<TP, VEC>*>(gamma + c);
            const LnVec<TP, VEC> b = *reinterpret_cast<const LnVec<TP, VEC>*>(beta + c);
            LnVec<TY, VEC> o;
#pragma unroll
            for (int e = 0; e < VEC; ++e) o.v[e] = from_acc<TY>(v[k][e] * rstd * to_acc(g.v[e]) + to_acc(b.v[e]));
            *reinterpret_cast<LnVec<TY, VEC>*>(y + row * D + c) = o;
        }
    }
    if (stats && sub == 0) stats[row] = mean, stats[N + row] = rstd;
}

// dx = rstd (g - mean(g) - xhat mean(g xhat)) + dres, g = dy * gamma; part [workgroup][2][D]: sums of dy * xhat and of dy.
// dx_copy: dx in dy's type for the 16-bit layer in front (219 000 x 48: 2 us here, a conversion of its own 11)
template <typename TX, typename TG, typename TP, int L, int V, bool EXACT>
__global__ __launch_bounds__(LN_THREADS) void layer_norm_backward_kernel(const TG* __restrict__ dy, const TX* __restrict__ x,
                                                                         const float* __restrict__ stats, int64_t N, int D,
                                                                         const TP* __restrict__ gamma,
                                                                         const TX* __restrict__ dres, TX* __restrict__ dx,
                                                                         float* __restrict__ part, TG* __restrict__ dx_copy) {
    constexpr int VEC = 16 / sizeof(TX), RPB = LN_THREADS / L;
    extern __shared__ float ln_sums[];                                   // [row slot RPB][2][D]
    const int sub = threadIdx.x % L, slot = threadIdx.x / L;
    const float inv = 1.f / (float)D;
    float gm[V][VEC], dg[V][VEC], db[V][VEC];
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int c = (k * L + sub) * VEC;
#pragma unroll
        for (int e = 0; e < VEC; ++e) gm[k][e] = dg[k][e] = db[k][e] = 0.f;
        if (EXACT || c < D) {
            const LnVec<TP, VEC> g = *reinterpret_cast<const LnVec<TP, VEC>*>(gamma + c);
#pragma unroll
            for (int e = 0; e < VEC; ++e) gm[k][e] = to_acc(g.v[e]);
        }
    }
    for (int64_t row = (int64_t)blockIdx.x * RPB + slot; row < N; row += (int64_t)gridDim.x * RPB) {
        const float mean = stats[row], rstd = stats[N + row];
        float xh[V][VEC], gy[V][VEC], s1 = 0.f, s2 = 0.f;
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const int c = (k * L + sub) * VEC;
            if (EXACT || c < D) {
                const LnVec<TX, VEC> px = *reinterpret_cast<const LnVec<TX, VEC>*>(x + row * D + c);
                const LnVec<TG, VEC> pg = *reinterpret_cast<const LnVec<TG, VEC>*>(dy + row * D + c);
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    const float d = to_acc(pg.v[e]);
                    xh[k][e] = (to_acc(px.v[e]) - mean) * rstd;
                    dg[k][e] += d * xh[k][e];
                    db[k][e] += d;
                    gy[k][e] = d * gm[k][e];
                    s1 += gy[k][e];
                    s2 += gy[k][e] * xh[k][e];
                }
            }
        }
        s1 = lanes_sum<L>(s1) * inv;
        s2 = lanes_sum<L>(s2) * inv;
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const int c = (k * L + sub) * VEC;
            if (EXACT || c < D) {
                LnVec<TX, VEC> r, o;
                if (dres) r = *reinterpret_cast<const LnVec<TX, VEC>*>(dres + row * D + c);
#pragma unroll
                for (int e = 0; e < VEC; ++e)
                    o.v[e] = from_acc<TX>(rstd * (gy[k][e] - s1 - xh[k][e] * s2) + (dres ? to_acc(r.v[e]) : 0.f));
                *reinterpret_cast<LnVec<TX, VEC>*>(dx + row * D + c) = o;
                if (dx_copy) {
                    LnVec<TG, VEC> half;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) half.v[e] = from_acc<TG>(to_acc(o.v[e]));
                    *reinterpret_cast<LnVec<TG, VEC>*>(dx_copy + row * D + c) = half;
                }
            }
        }
    }
    float* mine = ln_sums + slot * 2 * D;
#pragma unroll
    for (int k = 0; k < V; ++k) {
        const int c = (k * L + sub) * VEC;
        if (EXACT || c < D)
#pragma unroll
            for (int e = 0; e < VEC; ++e) mine[c + e] = dg[k][e], mine[D + c + e] = db[k][e];
    }
    __syncthreads();
    for (int c = threadIdx.x; c < 2 * D; c += LN_THREADS) {
        float s = 0.f;
        for (int r = 0; r < RPB; ++r) s += ln_sums[r * 2 * D + c];
        part[(int64_t)blockIdx.x * 2 * D + c] = s;
    }
}

// gamma / beta gradients: column sums of the partial sums.  A workgroup takes 4 columns, 64 threads share a column, each
// adds every 64th part in order, the 64 sums in a fixed tree (16 columns and 16 threads: 19 us for 1024 parts of 192)
template <typename TP>
__global__ __launch_bounds__(256) void layer_norm_sums_kernel(const float* __restrict__ part, int parts, int D,
                                                              TP* __restrict__ dgamma, TP* __restrict__ dbeta) {
    __shared__ float sums[64][5];
    const int cl = threadIdx.x & 3, pl = threadIdx.x >> 2, c = blockIdx.x * 4 + cl;
    float s = 0.f;
#pragma unroll 4
    for (int p = pl; p < parts; p += 64) s += part[(int64_t)p * 2 * D + c];
    sums[pl][cl] = s;
    __syncthreads();
#pragma unroll
    for (int w = 32; w >= 1; w >>= 1) {
        if (pl < w) sums[pl][cl] += sums[pl + w][cl];
        __syncthreads();
    }
    if (pl == 0) (c < D ? dgamma[c] : dbeta[c - D]) = from_acc<TP>(sums[0][cl]);
}

// lanes per row and pieces per lane for rows of `pieces` pieces of 16 bytes; false if a row is too long
static bool ln_split(int pieces, int* lanes, int* per_lane, bool* exact) {
    int p2 = 1;
    while (p2 < 64 && pieces % (2 * p2) == 0) p2 *= 2;
    if (p2 >= 4 && pieces / p2 <= 3) {
        *lanes = p2, *per_lane = pieces / p2, *exact = true;
        return true;
    }
    int l = 4;
    while (l < 64 && l < pieces) l *= 2;
    const int v = (pieces + l - 1) / l;
    *lanes = l, *per_lane = v <= 3 ? v : v <= 4 ? 4 : v <= 6 ? 6 : 8, *exact = *lanes * *per_lane == pieces;
    return v <= 8;
}

static int64_t ln_backward_blocks(int64_t N, int lanes) {
    const int rows = LN_THREADS / lanes;
    return std::min<int64_t>((N + rows - 1) / rows, 512);                // two workgroups per compute unit
}

template <typename TX, typename TO, typename TP, int L, int V, bool EXACT>
static void ln_launch(bool backward, const void* a, const void* b, int64_t N, int D, const void* gamma, const void* beta, float eps,
                      void* out, float* stats, const void* dres, float* part, void* copy, hipStream_t s) {
    if (!backward) {
        const int64_t blocks = (N + LN_THREADS / L - 1) / (LN_THREADS / L);
        hipLaunchKernelGGL((layer_norm_forward_kernel<TX, TO, TP, L, V, EXACT>), dim3((unsigned)blocks), dim3(LN_THREADS), 0, s,
                           static_cast<const TX*>(a), N, D, static_cast<const TP*>(gamma), static_cast<const TP*>(beta), eps,
                           static_cast<TO*>(out), stats);
    } else {
        const size_t lds = (size_t)(LN_THREADS / L) * 2 * D * sizeof(float);
        hipLaunchKernelGGL((layer_norm_backward_kernel<TX, TO, TP, L, V, EXACT>), dim3((unsigned)ln_backward_blocks(N, L)),
                           dim3(LN_THREADS), lds, s, static_cast<const TO*>(a), static_cast<const TX*>(b), stats, N, D,
                           static_cast<const TP*>(gamma), static_cast<const TX*>(dres), static_cast<TX*>(out), part, static_cast<TO*>(copy));
    }
}

template <typename TX, typename TO, typename TP>
static void ln_dispatch(bool backward, const void* a, const void* b, int64_t N, int D, const void* gamma, const void* beta, float eps,
                        void* out, float* stats, const void* dres, float* part, void* copy, hipStream_t s) {
    int lanes = 0, per = 0;
    bool exact = false;
    ln_split(D / (16 / (int)sizeof(TX)), &lanes, &per, &exact);
#define LN_CASE(L, V)                                                                                                       \
    if (lanes == L && per == V) {                                                                                           \
        exact ? ln_launch<TX, TO, TP, L, V, true>(backward, a, b, N, D, gamma, beta, eps, out, stats, dres, part, copy, s)  \
              : ln_launch<TX, TO, TP, L, V, false>(backward, a, b, N, D, gamma, beta, eps, out, stats, dres, part, copy, s);\
        return;                                                                                                             \
    }
    LN_CASE(4, 1) LN_CASE(4, 2) LN_CASE(4, 3) LN_CASE(8, 1) LN_CASE(8, 2) LN_CASE(8, 3) LN_CASE(16, 1) LN_CASE(16, 2)
    LN_CASE(16, 3) LN_CASE(32, 1) LN_CASE(32, 2) LN_CASE(32, 3) LN_CASE(64, 1) LN_CASE(64, 2) LN_CASE(64, 3) LN_CASE(64, 4)
    LN_CASE(64, 6) LN_CASE(64, 8)
#undef LN_CASE
}

// x dtype, other side's dtype (y, or dy) -> the instantiation; parameters are fp32 where x is, else of x's type
static int ln_run(bool backward, int x_dtype, int o_dtype, const void* a, const void* b, int64_t N, int D, const void* gamma,
                  const void* beta, float eps, void* out, float* stats, const void* dres, float* part, void* copy, hipStream_t s) {
#define LN_RUN(TX, TO, TP) ln_dispatch<TX, TO, TP>(backward, a, b, N, D, gamma, beta, eps, out, stats, dres, part, copy, s)
    if (x_dtype == SSWIN_F32 && o_dtype == SSWIN_F32) LN_RUN(float, float, float);
    else if (x_dtype == SSWIN_F32 && o_dtype == SSWIN_F16) LN_RUN(float, __half, float);
    else if (x_dtype == SSWIN_F32 && o_dtype == SSWIN_BF16) LN_RUN(float, __hip_bfloat16, float);
    else if (x_dtype == SSWIN_F16 && o_dtype == SSWIN_F16) LN_RUN(__half, __half, __half);
    else if (x_dtype == SSWIN_BF16 && o_dtype == SSWIN_BF16) LN_RUN(__hip_bfloat16, __hip_bfloat16, __hip_bfloat16);
    else return fail("layer_norm: x of type %d with the other side of type %d is not supported", x_dtype, o_dtype);
#undef LN_RUN
    return launch_ok("layer_norm");
}

}  // namespace sswin

using namespace sswin;

extern "C" {

int sswin_layer_norm_supported(int x_dtype, int D) {
    const int vec = x_dtype == SSWIN_F32 ? 4 : (x_dtype == SSWIN_F16 || x_dtype == SSWIN_BF16) ? 8 : 0;
    int l, v;
    bool e;
    return vec && D > 0 && D % vec == 0 && ln_split(D / vec, &l, &v, &e) &&
           (size_t)(LN_THREADS / l) * 2 * D * sizeof(float) <= 64 * 1024;      // the backward's sums of a workgroup
}

size_t sswin_layer_norm_backward_workspace_bytes(int x_dtype, int64_t N, int D) {
    if (N <= 0 || !sswin_layer_norm_supported(x_dtype, D)) return 0;
    int l, v;
    bool e;
    ln_split(D / (x_dtype == SSWIN_F32 ? 4 : 8), &l, &v, &e);
    return (size_t)ln_backward_blocks(N, l) * 2 * D * sizeof(float);
}

int sswin_layer_norm_forward(int x_dtype, int y_dtype, const void* x, int64_t N, int D, const void* gamma, const void* beta, float eps,
                             void* y, float* stats, void* stream) {
    SSWIN_CHECK(N >= 0, "layer_norm_forward: bad sizes");
    SSWIN_CHECK(sswin_layer_norm_supported(x_dtype, D), "layer_norm_forward: rows of %d values of type %d are not supported", D, x_dtype);
    if (N == 0) return 0;
    SSWIN_CHECK(x && gamma && beta && y, "layer_norm_forward: null pointer");
    SSWIN_CHECK(((uintptr_t)x | (uintptr_t)gamma | (uintptr_t)beta | (uintptr_t)y) % 16 == 0, "layer_norm_forward: pointers must be 16-byte aligned");
    return ln_run(false, x_dtype, y_dtype, x, nullptr, N, D, gamma, beta, eps, y, stats, nullptr, nullptr, nullptr, static_cast<hipStream_t>(stream));
}

int sswin_layer_norm_backward(int x_dtype, int dy_dtype, const void* dy, const void* x, const float* stats, int64_t N, int D,
                              const void* gamma, const void* dres, void* dx, void* dgamma, void* dbeta, void* ws, size_t ws_bytes,
                              void* stream) {
    return sswin_layer_norm_backward_copy(x_dtype, dy_dtype, dy, x, stats, N, D, gamma, dres, dx, nullptr, dgamma, dbeta, ws, ws_bytes, stream);
}

int sswin_layer_norm_backward_copy(int x_dtype, int dy_dtype, const void* dy, const void* x, const float* stats, int64_t N, int D,
                                   const void* gamma, const void* dres, void* dx, void* dx_copy, void* dgamma, void* dbeta, void* ws,
                                   size_t ws_bytes, void* stream) {
    SSWIN_CHECK(N > 0, "layer_norm_backward: bad sizes");
    SSWIN_CHECK(sswin_layer_norm_supported(x_dtype, D), "layer_norm_backward: rows of %d values of type %d are not supported", D, x_dtype);
    SSWIN_CHECK(dy && x && stats && gamma && dx && dgamma && dbeta && ws, "layer_norm_backward: null pointer");
    SSWIN_CHECK(((uintptr_t)dy | (uintptr_t)x | (uintptr_t)gamma | (uintptr_t)dres | (uintptr_t)dx | (uintptr_t)dx_copy | (uintptr_t)ws) % 16 == 0,
                "layer_norm_backward: pointers must be 16-byte aligned");
    SSWIN_CHECK(ws_bytes >= sswin_layer_norm_backward_workspace_bytes(x_dtype, N, D), "layer_norm_backward: workspace too small");
    hipStream_t s = static_cast<hipStream_t>(stream);
    float* part = static_cast<float*>(ws);
    if (int rc = ln_run(true, x_dtype, dy_dtype, dy, x, N, D, gamma, nullptr, 0.f, dx, const_cast<float*>(stats), dres, part, dx_copy, s)) return rc;
    int l, v;
    bool e;
    ln_split(D / (x_dtype == SSWIN_F32 ? 4 : 8), &l, &v, &e);
    const int parts = (int)ln_backward_blocks(N, l);
    const dim3 grid(2 * D / 4), block(256);
    if (x_dtype == SSWIN_F32)
        hipLaunchKernelGGL(layer_norm_sums_kernel<float>, grid, block, 0, s, part, parts, D, static_cast<float*>(dgamma), static_cast<float*>(dbeta));
    else if (x_dtype == SSWIN_F16)
        hipLaunchKernelGGL(layer_norm_sums_kernel<__half>, grid, block, 0, s, part, parts, D, static_cast<__half*>(dgamma), static_cast<__half*>(dbeta));
    else
        hipLaunchKernelGGL(layer_norm_sums_kernel<__hip_bfloat16>, grid, block, 0, s, part, parts, D, static_cast<__hip_bfloat16*>(dgamma),
                           static_cast<__hip_bfloat16*>(dbeta));
    return launch_ok("layer_norm_backward sums");
}

}  // extern "C"
