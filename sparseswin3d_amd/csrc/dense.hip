// Dense layers over all tokens (nn.Linear of sparse_swin/swin3d_base.py:606-610 and of the feed-forward part,
// :722-735), forward, input gradient and weight gradient, for fp32, fp16 and bf16 tokens, with what follows the
// product folded into its last step: bias, GELU and its derivative, the product with that derivative, the residual sum.
//
// Products run on the 16-bit matrix cores with fp32 accumulation.  fp32 operands are split exactly into three bf16
// pieces (x = h + m + l by truncation and exact subtraction) and a product is the sum of the six piece products that
// weigh at least 2^-16 of the leading one; what is dropped is below 2^-23 of the product.
//
// dense_rows_kernel: a workgroup of WM wavefronts owns BM = 32 MT WM rows and 96 columns.  Both operands pass through
// registers (conversion, splitting) into LDS in matrix operand order, [k step][row tile][plane][lane] pieces of 16
// bytes, so that every operand read is one conflict-free 16-byte read per lane; two buffers, one barrier per BK columns
// of the reduction, the next BK in flight meanwhile.  96 columns because every layer of a stage has a multiple of 48.
// The tile of the result goes back through LDS, so that bias, residual and result are touched in 16-byte pieces of whole
// row segments.
// dense_small_kernel: few rows and many channels (the deep stages): 32 x 32 tiles, the wavefronts of a workgroup share
// the reduction instead of the rows, so that a few hundred rows still put a wavefront on every SIMD.
// dense_wgrad_kernel: dW = dY^T X, db = column sums of dY: the reduction runs over the rows, both operands are read as
// 8 rows x 2 columns per lane and turned in registers.  Row chunks are added by a second kernel in a fixed order.
#include <math.h>

#include <algorithm>

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

template <typename T> __device__ __forceinline__ uint32_t pack2(float a, float b);
template <> __device__ __forceinline__ uint32_t pack2<__half>(float a, float b) {
    return (uint32_t)__half_as_ushort(__float2half(a)) | ((uint32_t)__half_as_ushort(__float2half(b)) << 16);
}
template <> __device__ __forceinline__ uint32_t pack2<__hip_bfloat16>(float a, float b) {
    const __hip_bfloat16 x = __float2bfloat16(a), y = __float2bfloat16(b);
    return (uint32_t)__builtin_bit_cast(uint16_t, x) | ((uint32_t)__builtin_bit_cast(uint16_t, y) << 16);
}

__device__ __forceinline__ void split2(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
    const uint32_t u0 = __builtin_bit_cast(uint32_t, x0), u1 = __builtin_bit_cast(uint32_t, x1);
    const float r0 = x0 - __builtin_bit_cast(float, u0 & 0xffff0000u), r1 = x1 - __builtin_bit_cast(float, u1 & 0xffff0000u);
    const uint32_t v0 = __builtin_bit_cast(uint32_t, r0), v1 = __builtin_bit_cast(uint32_t, r1);
    const float s0 = r0 - __builtin_bit_cast(float, v0 & 0xffff0000u), s1 = r1 - __builtin_bit_cast(float, v1 & 0xffff0000u);
    h = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
    m = __builtin_amdgcn_perm(v1, v0, 0x07060302u);
    l = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, s1), __builtin_bit_cast(uint32_t, s0), 0x07060302u);
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

// ------------------------------------------------------------------------------------------
// Raw values of a unit on their way from memory to LDS.
// Along: 8 consecutive values of one row (reduction along the row).  Down: 8 rows x 2 columns (reduction down the rows).
// ------------------------------------------------------------------------------------------
template <typename T, typename TS> struct Along {
    static constexpr bool WIDE = sizeof(TS) == 4;
    u32x4 r[WIDE ? 2 : 1];
    __device__ __forceinline__ void load(const TS* p) {
        r[0] = *reinterpret_cast<const u32x4*>(p);
        if constexpr (WIDE) r[1] = *reinterpret_cast<const u32x4*>(p + 4);
    }
    __device__ __forceinline__ void zero() {
        r[0] = u32x4{0, 0, 0, 0};
        if constexpr (WIDE) r[1] = u32x4{0, 0, 0, 0};
    }
    __device__ __forceinline__ void planes(u32x4 (&out)[Op<T>::PL]) const {
        if constexpr (!WIDE) {
            out[0] = r[0];
        } else {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = __builtin_bit_cast(float, e < 4 ? r[0][e] : r[1][e - 4]);
            planes_of<T>(v, out);
        }
    }
};

template <typename T, typename TS> struct Down {
    static constexpr bool WIDE = sizeof(TS) == 4;
    uint32_t r[8][WIDE ? 2 : 1];
    __device__ __forceinline__ void load(int e, const TS* p) {
        r[e][0] = reinterpret_cast<const uint32_t*>(p)[0];
        if constexpr (WIDE) r[e][1] = reinterpret_cast<const uint32_t*>(p)[1];
    }
    __device__ __forceinline__ void zero(int e) {
        r[e][0] = 0;
        if constexpr (WIDE) r[e][1] = 0;
    }
    // column c (0 or 1) of the pair
    __device__ __forceinline__ void planes(int c, u32x4 (&out)[Op<T>::PL]) const {
        if constexpr (WIDE) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = __builtin_bit_cast(float, r[e][c]);
            planes_of<T>(v, out);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) out[0][q] = __builtin_amdgcn_perm(r[2 * q + 1][0], r[2 * q][0], c ? 0x07060302u : 0x05040100u);
        }
    }
    __device__ __forceinline__ float sum(int c) const;
};
template <typename T> __device__ __forceinline__ float half_of(uint32_t w, int c);
template <> __device__ __forceinline__ float half_of<__half>(uint32_t w, int c) {
    return __half2float(__ushort_as_half((unsigned short)(c ? w >> 16 : w & 0xffffu)));
}
template <> __device__ __forceinline__ float half_of<__hip_bfloat16>(uint32_t w, int c) {
    return __builtin_bit_cast(float, c ? w & 0xffff0000u : w << 16);
}
template <typename T, typename TS> __device__ __forceinline__ float Down<T, TS>::sum(int c) const {
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        if constexpr (WIDE) s += __builtin_bit_cast(float, r[e][c]);
        else s += half_of<T>(r[e][0], c);
    }
    return s;
}

// position of (row, 8-value chunk) inside its 32-row operand block: the rows of a chunk are rotated by the chunk, so
// that lanes which hold the chunks of one row write to different banks
template <int BK> __device__ __forceinline__ int swz(int chunk) { return BK == 16 ? (chunk & 1) * 4 : chunk & 7; }

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

// ------------------------------------------------------------------------------------------
// y [N, P] = last step of x [N, K] Wop, Wop [K, P] = W^T of W [P, K] (DOWN = false) or W [K, P] itself (DOWN = true)
// ------------------------------------------------------------------------------------------
template <typename T, typename TB, typename TO, int EPI, bool DOWN, int WM, int MT, int OCC>
__global__ __launch_bounds__(WM * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void dense_rows_kernel(const T* __restrict__ x, int64_t N, int K, const TB* __restrict__ w, int P,
                                                             int groups, Epilogue ep) {
    constexpr int PL = Op<T>::PL, BK = PL == 3 ? 16 : 48, KS = BK / 16, KC = BK / 8;
    constexpr int NT = 3, BN = 96, BM = WM * MT * 32, THREADS = WM * 64;
    constexpr int A_UNITS = BM * KC, UA = (A_UNITS + THREADS - 1) / THREADS;
    constexpr int B_UNITS = (DOWN ? BN / 2 : BN) * KC, UB = (B_UNITS + THREADS - 1) / THREADS;
    constexpr int A_LDS = KS * (BM / 32) * PL * 64, B_LDS = KS * NT * PL * 64, BUF = A_LDS + B_LDS;      // 16-byte pieces
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    int cg;
    int64_t rb;
    block_of(groups, cg, rb);
    const int64_t row0 = rb * BM;
    const int col0 = cg * BN;

    // addresses: a uniform base that moves along the reduction plus 32-bit lane offsets formed once
    Along<T, T> ra[UA];
    typename std::conditional<DOWN, Down<T, TB>, Along<T, TB>>::type rw[UB];
    uint32_t oa[UA], ow[UB];
    const int last = (int)(N - 1 - row0 < BM - 1 ? N - 1 - row0 : BM - 1);   // rows past the end repeat the last one
#pragma unroll
    for (int i = 0; i < UA; ++i) {
        const int u = threadIdx.x + i * THREADS;
        oa[i] = (uint32_t)(min(u / KC, last) * K + (u % KC) * 8);
    }
#pragma unroll
    for (int i = 0; i < UB; ++i) {
        const int u = threadIdx.x + i * THREADS;
        if (DOWN) ow[i] = (uint32_t)((u / (BN / 2)) * 8 * P + min(col0 + (u % (BN / 2)) * 2, P - 2));
        else ow[i] = (uint32_t)(min(col0 + u / KC, P - 1) * K + (u % KC) * 8);
    }
    const T* xb = x + row0 * K;
    auto request = [&](int k0) {
#pragma unroll
        for (int i = 0; i < UA; ++i) {
            const int u = threadIdx.x + i * THREADS;
            if (A_UNITS % THREADS == 0 || u < A_UNITS) {
                if (BK == 16 || k0 + (u % KC) * 8 < K) ra[i].load(xb + k0 + oa[i]);
                else ra[i].zero();
            }
        }
#pragma unroll
        for (int i = 0; i < UB; ++i) {
            const int u = threadIdx.x + i * THREADS;
            if (B_UNITS % THREADS == 0 || u < B_UNITS) {
                if constexpr (DOWN) {
                    const bool in = BK == 16 || k0 + (u / (BN / 2)) * 8 < K;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        if (in) rw[i].load(e, w + (int64_t)(k0 + e) * P + ow[i]);
                        else rw[i].zero(e);
                    }
                } else {
                    if (BK == 16 || k0 + (u % KC) * 8 < K) rw[i].load(w + k0 + ow[i]);
                    else rw[i].zero();
                }
            }
        }
    };
    auto put = [&](u32x4* base, int tiles, int row, int c, const u32x4 (&p)[PL]) {
        u32x4* dst = base + (((c >> 1) * tiles + (row >> 5)) * PL) * 64 + (c & 1) * 32 + ((row & 31) ^ swz<BK>(c));
#pragma unroll
        for (int q = 0; q < PL; ++q) dst[q * 64] = p[q];
    };
    auto store = [&](u32x4* buf) {
#pragma unroll
        for (int i = 0; i < UA; ++i) {
            const int u = threadIdx.x + i * THREADS;
            if (A_UNITS % THREADS == 0 || u < A_UNITS) {
                u32x4 p[PL];
                ra[i].planes(p);
                put(buf, BM / 32, u / KC, u % KC, p);
            }
        }
#pragma unroll
        for (int i = 0; i < UB; ++i) {
            const int u = threadIdx.x + i * THREADS;
            if (B_UNITS % THREADS == 0 || u < B_UNITS) {
                u32x4 p[PL];
                if constexpr (DOWN) {
                    rw[i].planes(0, p);
                    put(buf + A_LDS, NT, (u % (BN / 2)) * 2, u / (BN / 2), p);
                    rw[i].planes(1, p);
                    put(buf + A_LDS, NT, (u % (BN / 2)) * 2 + 1, u / (BN / 2), p);
                } else {
                    rw[i].planes(p);
                    put(buf + A_LDS, NT, u / KC, u % KC, p);
                }
            }
        }
    };

    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const int nk = (K + BK - 1) / BK;
    request(0);
    store(lds);
    for (int kb = 0; kb < nk; ++kb) {
        __syncthreads();
        if (kb + 1 < nk) request((kb + 1) * BK);
        const u32x4* buf = lds + (kb & 1) * BUF;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int at = half * 32 + (l32 ^ swz<BK>(ks * 2 + half));
            u32x4 a[MT][PL], b[NT][PL];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int q = 0; q < PL; ++q) a[i][q] = buf[((ks * (BM / 32) + wave * MT + i) * PL + q) * 64 + at];
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < PL; ++q) b[j][q] = buf[A_LDS + ((ks * NT + j) * PL + q) * 64 + at];
#pragma unroll
            for (int p = 0; p < Op<T>::NP; ++p)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = Op<T>::mfma(a[i][Op<T>::PA[p]], b[j][Op<T>::PB[p]], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);                           // operands of later steps stay out of registers
        }
        if (kb + 1 < nk) store(lds + ((kb + 1) & 1) * BUF);
    }
    // the tile of the wavefront, 32 rows at a time, through its own part of LDS (pitch 100: rows start 4 banks apart)
    __syncthreads();
    constexpr int PITCH = BN + 4;
    float* mine = reinterpret_cast<float*>(lds) + wave * 32 * PITCH;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int64_t r0 = row0 + (wave * MT + i) * 32;
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) mine[acc_row(r, half) * PITCH + j * 32 + l32] = acc[i][j][r];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < 32 * (BN / 4) / 64; ++q) {
            const int e = q * 64 + lane, rr = e / (BN / 4), cc = (e % (BN / 4)) * 4;
            const f32x4 v = *reinterpret_cast<const f32x4*>(mine + rr * PITCH + cc);
            if (r0 + rr < N && col0 + cc < P) finish4<T, TB, TO, EPI>(ep, r0 + rr, col0 + cc, P, v);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ------------------------------------------------------------------------------------------
// The same for few rows: a workgroup owns a 32 x 32 tile, its 8 wavefronts take every 8th 16-wide step of the reduction
// and add their tiles through LDS in a fixed order.
// ------------------------------------------------------------------------------------------
constexpr int SMALL_WAVES = 8;
template <typename T, typename TB, typename TO, int EPI, bool DOWN>
__global__ __launch_bounds__(SMALL_WAVES * 64) void dense_small_kernel(const T* __restrict__ x, int64_t N, int K, const TB* __restrict__ w, int P,
                                                                    int groups, Epilogue ep) {
    constexpr int PL = Op<T>::PL;
    __shared__ __attribute__((aligned(16))) float sums[SMALL_WAVES][32 * 36];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int cg = blockIdx.x % groups;
    const int64_t row0 = (int64_t)(blockIdx.x / groups) * 32;
    const int col0 = cg * 32, steps = K / 16;
    const int64_t row = row0 + l32 < N ? row0 + l32 : N - 1;
    const int col = min(col0 + l32, P - 1);
    const T* xp = x + row * K + half * 8;
    f32x16 acc = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    constexpr int AHEAD = 3;                                             // steps of a wavefront in flight
    Along<T, T> ra[AHEAD];
    Along<T, TB> rb[DOWN ? 1 : AHEAD];
    float vb[DOWN ? AHEAD : 1][8];
    auto request = [&](int slot, int s) {
        ra[slot].load(xp + s * 16);
        if constexpr (DOWN) {
#pragma unroll
            for (int e = 0; e < 8; ++e) vb[slot][e] = to_acc(w[(int64_t)(s * 16 + half * 8 + e) * P + col]);
        } else {
            rb[slot].load(w + (int64_t)col * K + s * 16 + half * 8);
        }
    };
#pragma unroll
    for (int q = 0; q < AHEAD; ++q)
        if (wave + q * SMALL_WAVES < steps) request(q, wave + q * SMALL_WAVES);
    for (int s0 = wave; s0 < steps; s0 += AHEAD * SMALL_WAVES) {
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) {
            const int s = s0 + q * SMALL_WAVES;
            if (s < steps) {
                u32x4 a[PL], b[PL];
                ra[q].planes(a);
                if constexpr (DOWN) planes_of<T>(vb[q], b);
                else rb[q].planes(b);
                if (s + AHEAD * SMALL_WAVES < steps) request(q, s + AHEAD * SMALL_WAVES);
#pragma unroll
                for (int p = 0; p < Op<T>::NP; ++p) acc = Op<T>::mfma(a[Op<T>::PA[p]], b[Op<T>::PB[p]], acc);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) sums[wave][acc_row(r, half) * 36 + l32] = acc[r];
    __syncthreads();
    if (threadIdx.x < 256) {
        const int rr = threadIdx.x >> 3, cc = (threadIdx.x & 7) * 4;
        f32x4 v = *reinterpret_cast<const f32x4*>(&sums[0][rr * 36 + cc]);
#pragma unroll
        for (int q = 1; q < SMALL_WAVES; ++q) v += *reinterpret_cast<const f32x4*>(&sums[q][rr * 36 + cc]);
        if (row0 + rr < N && col0 + cc < P) finish4<T, TB, TO, EPI>(ep, row0 + rr, col0 + cc, P, v);
    }
}

// ------------------------------------------------------------------------------------------
// dW [P, K] = dY^T X, db [P] = column sums of dY.  A workgroup owns BM x BN of dW for one chunk of rows.
// ------------------------------------------------------------------------------------------
template <typename T, int WM, int WN, int MT, int NT, int OCC>
__global__ __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void dense_wgrad_kernel(const T* __restrict__ dy, const T* __restrict__ x, int64_t N, int P, int K,
                                                                   int tiles_p, int tiles_k, int64_t rows_per_chunk, float* __restrict__ part_w,
                                                                   float* __restrict__ part_b) {
    constexpr int PL = Op<T>::PL, BK = PL == 3 ? 16 : 32, KS = BK / 16, KC = BK / 8;
    constexpr int BM = WM * MT * 32, BN = WN * NT * 32, THREADS = WM * WN * 64;
    constexpr int A_UNITS = BM / 2 * KC, UA = (A_UNITS + THREADS - 1) / THREADS;
    constexpr int B_UNITS = BN / 2 * KC, UB = (B_UNITS + THREADS - 1) / THREADS;
    constexpr int A_LDS = KS * (BM / 32) * PL * 64, B_LDS = KS * (BN / 32) * PL * 64, BUF = A_LDS + B_LDS;
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int wm = wave / WN, wn = wave % WN;
    int tile;
    int64_t chunk;
    block_of(tiles_p * tiles_k, tile, chunk);
    const int p0 = (tile / tiles_k) * BM, k0 = (tile % tiles_k) * BN;
    const int64_t begin = chunk * rows_per_chunk, end = begin + rows_per_chunk < N ? begin + rows_per_chunk : N;
    const bool sums_here = part_b && k0 == 0;

    Down<T, T> ra[UA], rx[UB];
    float bs[UA][2];
#pragma unroll
    for (int i = 0; i < UA; ++i) bs[i][0] = bs[i][1] = 0.f;
    uint32_t oa[UA], ox[UB];
#pragma unroll
    for (int i = 0; i < UA; ++i) {
        const int u = threadIdx.x + i * THREADS;
        oa[i] = (uint32_t)((u / (BM / 2)) * 8 * P + min(p0 + (u % (BM / 2)) * 2, P - 2));
    }
#pragma unroll
    for (int i = 0; i < UB; ++i) {
        const int u = threadIdx.x + i * THREADS;
        ox[i] = (uint32_t)((u / (BN / 2)) * 8 * K + min(k0 + (u % (BN / 2)) * 2, K - 2));
    }
    auto request = [&](int64_t n0) {
        const T* yb = dy + n0 * P;
        const T* xb = x + n0 * K;
        if (n0 + BK <= end) {
#pragma unroll
            for (int i = 0; i < UA; ++i)
                if (A_UNITS % THREADS == 0 || (int)threadIdx.x + i * THREADS < A_UNITS)
#pragma unroll
                    for (int e = 0; e < 8; ++e) ra[i].load(e, yb + e * P + oa[i]);
#pragma unroll
            for (int i = 0; i < UB; ++i)
                if (B_UNITS % THREADS == 0 || (int)threadIdx.x + i * THREADS < B_UNITS)
#pragma unroll
                    for (int e = 0; e < 8; ++e) rx[i].load(e, xb + e * K + ox[i]);
        } else {                                                         // the ragged end of the rows: zeros past it
            const int left = (int)(end - n0);
#pragma unroll
            for (int i = 0; i < UA; ++i) {
                const int u = threadIdx.x + i * THREADS, n = (u / (BM / 2)) * 8;
                if (A_UNITS % THREADS == 0 || u < A_UNITS)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        if (n + e < left) ra[i].load(e, yb + e * P + oa[i]);
                        else ra[i].zero(e);
                    }
            }
#pragma unroll
            for (int i = 0; i < UB; ++i) {
                const int u = threadIdx.x + i * THREADS, n = (u / (BN / 2)) * 8;
                if (B_UNITS % THREADS == 0 || u < B_UNITS)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        if (n + e < left) rx[i].load(e, xb + e * K + ox[i]);
                        else rx[i].zero(e);
                    }
            }
        }
    };
    auto put = [&](u32x4* base, int tiles, int row, int c, const u32x4 (&p)[PL]) {
        u32x4* dst = base + (((c >> 1) * tiles + (row >> 5)) * PL) * 64 + (c & 1) * 32 + (row & 31);
#pragma unroll
        for (int q = 0; q < PL; ++q) dst[q * 64] = p[q];
    };
    auto store = [&](u32x4* buf) {
#pragma unroll
        for (int i = 0; i < UA; ++i) {
            const int u = threadIdx.x + i * THREADS, pair = u % (BM / 2), c = u / (BM / 2);
            if (A_UNITS % THREADS == 0 || u < A_UNITS) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    u32x4 p[PL];
                    ra[i].planes(h, p);
                    put(buf, BM / 32, pair * 2 + h, c, p);
                    if (sums_here) bs[i][h] += ra[i].sum(h);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < UB; ++i) {
            const int u = threadIdx.x + i * THREADS, pair = u % (BN / 2), c = u / (BN / 2);
            if (B_UNITS % THREADS == 0 || u < B_UNITS) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    u32x4 p[PL];
                    rx[i].planes(h, p);
                    put(buf + A_LDS, BN / 32, pair * 2 + h, c, p);
                }
            }
        }
    };
    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const int nk = (int)((end - begin + BK - 1) / BK);
    request(begin);
    store(lds);
    for (int kb = 0; kb < nk; ++kb) {
        __syncthreads();
        if (kb + 1 < nk) request(begin + (int64_t)(kb + 1) * BK);
        const u32x4* buf = lds + (kb & 1) * BUF;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            u32x4 a[MT][PL], b[NT][PL];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int q = 0; q < PL; ++q) a[i][q] = buf[((ks * (BM / 32) + wm * MT + i) * PL + q) * 64 + lane];
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < PL; ++q) b[j][q] = buf[A_LDS + ((ks * (BN / 32) + wn * NT + j) * PL + q) * 64 + lane];
#pragma unroll
            for (int p = 0; p < Op<T>::NP; ++p)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = Op<T>::mfma(a[i][Op<T>::PA[p]], b[j][Op<T>::PB[p]], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);                           // operands of later steps stay out of registers
        }
        if (kb + 1 < nk) store(lds + ((kb + 1) & 1) * BUF);
    }
    float* pw = part_w + chunk * (int64_t)P * K;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int p = p0 + (wm * MT + i) * 32 + acc_row(r, half), k = k0 + (wn * NT + j) * 32 + l32;
                if (p < P && k < K) pw[(int64_t)p * K + k] = acc[i][j][r];
            }
    if (sums_here) {
        // unit u holds rows of chunk u / (BM / 2) of its column pair: the chunks of a pair are added in order
        __syncthreads();
        float* red = reinterpret_cast<float*>(lds);
#pragma unroll
        for (int i = 0; i < UA; ++i) {
            const int u = threadIdx.x + i * THREADS;
            if (A_UNITS % THREADS == 0 || u < A_UNITS) red[u * 2] = bs[i][0], red[u * 2 + 1] = bs[i][1];
        }
        __syncthreads();
        for (int c = threadIdx.x; c < BM; c += THREADS) {
            float s = 0.f;
#pragma unroll
            for (int q = 0; q < KC; ++q) s += red[(q * (BM / 2) + c / 2) * 2 + (c & 1)];
            if (p0 + c < P) part_b[chunk * P + p0 + c] = s;
        }
    }
}

// The same for few rows: a workgroup owns a 32 x 32 tile of dW, its 8 wavefronts take every 8th step of 16 rows and add
// their tiles through LDS in a fixed order, so that the result leaves in one launch.
template <typename T, typename TO>
__global__ __launch_bounds__(SMALL_WAVES * 64) void dense_wgrad_small_kernel(const T* __restrict__ dy, const T* __restrict__ x, int64_t N, int P, int K,
                                                                             int tiles_k, TO* __restrict__ dw, TO* __restrict__ db) {
    constexpr int PL = Op<T>::PL, AHEAD = 2;
    __shared__ __attribute__((aligned(16))) float sums[SMALL_WAVES][32 * 36];
    __shared__ float colsum[SMALL_WAVES][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int p0 = (int)(blockIdx.x / tiles_k) * 32, k0 = (int)(blockIdx.x % tiles_k) * 32;
    const int pc = min(p0 + l32, P - 1), kc = min(k0 + l32, K - 1), steps = (int)((N + 15) / 16);
    float va[AHEAD][8], vb[AHEAD][8], bsum = 0.f;
    auto request = [&](int slot, int s) {
        const int64_t n0 = (int64_t)s * 16 + half * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const bool in = n0 + e < N;
            va[slot][e] = in ? to_acc(dy[(n0 + e) * P + pc]) : 0.f;
            vb[slot][e] = in ? to_acc(x[(n0 + e) * K + kc]) : 0.f;
        }
    };
    f32x16 acc = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < AHEAD; ++q)
        if (wave + q * SMALL_WAVES < steps) request(q, wave + q * SMALL_WAVES);
    for (int s0 = wave; s0 < steps; s0 += AHEAD * SMALL_WAVES) {
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) {
            const int s = s0 + q * SMALL_WAVES;
            if (s < steps) {
                u32x4 a[PL], b[PL];
                planes_of<T>(va[q], a);
                planes_of<T>(vb[q], b);
#pragma unroll
                for (int e = 0; e < 8; ++e) bsum += va[q][e];
                if (s + AHEAD * SMALL_WAVES < steps) request(q, s + AHEAD * SMALL_WAVES);
#pragma unroll
                for (int p = 0; p < Op<T>::NP; ++p) acc = Op<T>::mfma(a[Op<T>::PA[p]], b[Op<T>::PB[p]], acc);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) sums[wave][acc_row(r, half) * 36 + l32] = acc[r];
    colsum[wave][lane] = bsum;
    __syncthreads();
    if (threadIdx.x < 256) {
        const int rr = threadIdx.x >> 3, cc = (threadIdx.x & 7) * 4;
        f32x4 v = *reinterpret_cast<const f32x4*>(&sums[0][rr * 36 + cc]);
#pragma unroll
        for (int q = 1; q < SMALL_WAVES; ++q) v += *reinterpret_cast<const f32x4*>(&sums[q][rr * 36 + cc]);
        if (p0 + rr < P && k0 + cc < K) {
            Vec4<TO> o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o.v[e] = from_acc<TO>(v[e]);
            *reinterpret_cast<Vec4<TO>*>(dw + (int64_t)(p0 + rr) * K + k0 + cc) = o;
        }
    } else if (db && k0 == 0 && threadIdx.x < 288 && p0 + (int)threadIdx.x - 256 < P) {
        float v = 0.f;
        const int c = threadIdx.x - 256;
#pragma unroll
        for (int q = 0; q < SMALL_WAVES; ++q) v += colsum[q][c] + colsum[q][c + 32];
        db[p0 + c] = from_acc<TO>(v);
    }
}

// out[e] = sum over chunks of part[chunk][e] for the weights and the bias behind each other; a block takes 16 x 4
// outputs, 16 threads share an output, each adds every 16th chunk in order, the 16 sums in a fixed tree
template <typename TO>
__global__ __launch_bounds__(256) void dense_wgrad_sum_kernel(const float* __restrict__ part_w, const float* __restrict__ part_b, int chunks,
                                                              int64_t PK, int P, TO* __restrict__ dw, TO* __restrict__ db) {
    __shared__ f32x4 sums[16][17];
    const int el = threadIdx.x & 15, cl = threadIdx.x >> 4;
    const int64_t e = ((int64_t)blockIdx.x * 16 + el) * 4;
    const bool weight = e < PK, valid = weight || (db && e - PK < P);
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    if (valid) {
        const float* src = weight ? part_w + e : part_b + (e - PK);
        const int64_t pitch = weight ? PK : P;
        for (int c = cl; c < chunks; c += 16) sum += *reinterpret_cast<const f32x4*>(src + c * pitch);
    }
    sums[cl][el] = sum;
    __syncthreads();
#pragma unroll
    for (int w = 8; w >= 1; w >>= 1) {
        if (cl < w) sums[cl][el] += sums[cl + w][el];
        __syncthreads();
    }
    if (cl == 0 && valid) {
        Vec4<TO> o;
#pragma unroll
        for (int q = 0; q < 4; ++q) o.v[q] = from_acc<TO>(sums[0][el][q]);
        *reinterpret_cast<Vec4<TO>*>(weight ? dw + e : db + (e - PK)) = o;
    }
}

// ------------------------------------------------------------------------------------------
// launches
// ------------------------------------------------------------------------------------------
static int device_cus() {
    static int cached = 0;
    if (!cached) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached = n;
    }
    return cached;
}

template <typename F> static int allow_lds(F* kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        SSWIN_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    return 0;
}

template <typename T, typename TB, typename TO, int EPI, bool DOWN, int WM, int MT, int OCC>
static int launch_rows(const T* x, int64_t N, int K, const TB* w, int P, const Epilogue& ep, hipStream_t s) {
    constexpr int PL = Op<T>::PL, BK = PL == 3 ? 16 : 48, BM = WM * MT * 32;
    constexpr size_t tiles = 2 * (size_t)(BK / 16) * (BM / 32 + 3) * PL * 64 * 16, out = (size_t)WM * 32 * 100 * 4;
    constexpr size_t bytes = tiles > out ? tiles : out;
    auto* k = dense_rows_kernel<T, TB, TO, EPI, DOWN, WM, MT, OCC>;
    static const int configured = allow_lds(k, bytes);
    if (configured) return configured;
    const int groups = (P + 95) / 96;
    const int64_t blocks = (N + BM - 1) / BM * groups;
    SSWIN_CHECK(blocks < (1ll << 31), "dense: too many rows");
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(WM * 64), bytes, s, x, N, K, w, P, groups, ep);
    return launch_ok("dense");
}

template <typename T, typename TB, typename TO, int EPI, bool DOWN>
static int launch_forward(const void* x, int64_t N, int K, const void* w, int P, const Epilogue& ep, hipStream_t s) {
    const T* xp = static_cast<const T*>(x);
    const TB* wp = static_cast<const TB*>(w);
    const int64_t small_blocks = (N + 31) / 32 * ((P + 31) / 32);
    // 128-row workgroups hide the latency of a step only from about 150 of them on: bf16 384 -> 1152 at 300 rows 5.3 us in 32 x 32
    // tiles and 10.7 here, at 2000 rows (192 workgroups) 15.9 and 11.6; fp32 96 -> 96 at 8000 rows (63) 5.7 and 9.5, at 16000 equal
    if ((N + 127) / 128 * ((P + 95) / 96) < 150 && small_blocks < (1ll << 31)) {
        hipLaunchKernelGGL((dense_small_kernel<T, TB, TO, EPI, DOWN>), dim3((unsigned)small_blocks), dim3(SMALL_WAVES * 64), 0, s, xp, N, K, wp, P,
                           (P + 31) / 32, ep);
        return launch_ok("dense, few rows");
    }
    // fp32 and 96 channels: the kernel that keeps Wop in LDS (219 000 rows, 96 -> 288: 89 us against 120 here, with a residual 133
    // and 202)
    if constexpr (Op<T>::PL == 3)
        if (K == 96 && P % 96 == 0) return staged_layer_96(xp, N, wp, P, DOWN, EPI, ep, s);
    // wavefronts per SIMD: what the registers allow without spilling (four: forward equal, input gradient 89 us against 40)
    return launch_rows<T, TB, TO, EPI, DOWN, 4, 1, 3>(xp, N, K, wp, P, ep, s);
}

template <typename T, typename TB, typename TO>
static int pick_forward(int epi, bool down, const void* x, int64_t N, int K, const void* w, int P, const Epilogue& ep, hipStream_t s) {
    if (down) {
        if (epi == EPI_NONE) return launch_forward<T, TB, TO, EPI_NONE, true>(x, N, K, w, P, ep, s);
        return launch_forward<T, TB, TO, EPI_SCALE, true>(x, N, K, w, P, ep, s);
    }
    if (epi == EPI_NONE) return launch_forward<T, TB, TO, EPI_NONE, false>(x, N, K, w, P, ep, s);
    if (epi == EPI_GELU) return launch_forward<T, TB, TO, EPI_GELU, false>(x, N, K, w, P, ep, s);
    return launch_forward<T, TB, TO, EPI_RESIDUAL, false>(x, N, K, w, P, ep, s);
}

// tiles of dW and row chunks: about `per_cu` workgroups per compute unit
struct WgradPlan {
    int tiles_p, tiles_k, chunks;
    int64_t rows;
};
static WgradPlan wgrad_plan(int64_t N, int P, int K, int bk, int bm, int bn, int per_cu) {
    WgradPlan p;
    p.tiles_p = (P + bm - 1) / bm;
    p.tiles_k = (K + bn - 1) / bn;
    const int64_t want = std::max<int64_t>(1, (int64_t)per_cu * device_cus() / ((int64_t)p.tiles_p * p.tiles_k));
    int64_t rows = std::max<int64_t>((N + want - 1) / want, 4 * bk);
    rows = (rows + bk - 1) / bk * bk;
    p.rows = rows;
    p.chunks = (int)((N + rows - 1) / rows);
    return p;
}

// rows up to which one launch of 32 x 32 tiles beats row chunks and their sums (284 rows 384 -> 1152: 19 us in chunks)
constexpr int64_t WGRAD_SMALL_ROWS = 1024;
// 128 x 192 tiles where dW has that many columns, otherwise 96 x 96 with more workgroups per compute unit: bf16, 219 000 rows
// 96 -> 288: 48 us in 96 x 96, 73 in 128 x 192; 8 119 rows 768 -> 2304: 107 and 77; fp32 35 569 rows 192 -> 576: 91 and 78
static bool wgrad_large(int K) { return K >= 192; }
static WgradPlan wgrad_plan(int dtype, int64_t N, int P, int K) {
    const int bk = dtype == SSWIN_F32 ? 16 : 32;
    return wgrad_large(K) ? wgrad_plan(N, P, K, bk, 128, 192, 2) : wgrad_plan(N, P, K, bk, 96, 96, 4);
}

template <typename T, typename TO, int WM, int WN, int MT, int NT, int OCC>
static int launch_wgrad_as(const WgradPlan& pl, const void* dy, const void* x, int64_t N, int P, int K, void* dw, void* db, float* ws, hipStream_t s) {
    constexpr int PL = Op<T>::PL, BK = PL == 3 ? 16 : 32;
    constexpr size_t bytes = 2 * (size_t)(BK / 16) * (WM * MT + WN * NT) * PL * 64 * 16;
    auto* k = dense_wgrad_kernel<T, WM, WN, MT, NT, OCC>;
    static const int configured = allow_lds(k, bytes);
    if (configured) return configured;
    float* part_b = ws + (size_t)pl.chunks * P * K;
    hipLaunchKernelGGL(k, dim3((unsigned)(pl.tiles_p * pl.tiles_k * pl.chunks)), dim3(WM * WN * 64), bytes, s, static_cast<const T*>(dy),
                       static_cast<const T*>(x), N, P, K, pl.tiles_p, pl.tiles_k, pl.rows, ws, db ? part_b : nullptr);
    if (int rc = launch_ok("dense weight gradient")) return rc;
    const int64_t PK = (int64_t)P * K;
    hipLaunchKernelGGL((dense_wgrad_sum_kernel<TO>), dim3((unsigned)((PK + P + 63) / 64)), dim3(256), 0, s, ws, part_b, pl.chunks, PK, P,
                       static_cast<TO*>(dw), static_cast<TO*>(db));
    return launch_ok("dense weight gradient, sums");
}

template <typename T, typename TO>
static int launch_wgrad(const void* dy, const void* x, int64_t N, int P, int K, void* dw, void* db, float* ws, hipStream_t s) {
    if (N <= WGRAD_SMALL_ROWS) {
        const int tp = (P + 31) / 32, tk = (K + 31) / 32;
        hipLaunchKernelGGL((dense_wgrad_small_kernel<T, TO>), dim3((unsigned)(tp * tk)), dim3(SMALL_WAVES * 64), 0, s, static_cast<const T*>(dy),
                           static_cast<const T*>(x), N, P, K, tk, static_cast<TO*>(dw), static_cast<TO*>(db));
        return launch_ok("dense weight gradient, few rows");
    }
    const WgradPlan pl = wgrad_plan(Op<T>::PL == 3 ? SSWIN_F32 : SSWIN_F16, N, P, K);
    if (wgrad_large(K)) return launch_wgrad_as<T, TO, 2, 2, 2, 3, 2>(pl, dy, x, N, P, K, dw, db, ws, s);
    return launch_wgrad_as<T, TO, 3, 1, 1, 3, 3>(pl, dy, x, N, P, K, dw, db, ws, s);
}

}  // namespace dense
}  // namespace sswin

using namespace sswin;
using namespace sswin::dense;

extern "C" {

int sswin_dense_supported(int dtype, int P, int K) {
    return (dtype == SSWIN_F32 || dtype == SSWIN_F16 || dtype == SSWIN_BF16) && P > 0 && K > 0 && P % 16 == 0 && K % 16 == 0;
}

int sswin_dense_forward(int dtype, int w_dtype, int out_dtype, int transposed, int epilogue, const void* x, int64_t N, int K, const void* w, const void* bias,
                        int P, const void* extra, void* y, void* slope, void* stream) {
    SSWIN_CHECK(N >= 0, "dense_forward: bad sizes");
    SSWIN_CHECK(sswin_dense_supported(dtype, P, K), "dense_forward: %d -> %d channels of type %d are not supported (multiples of 16)", K, P, dtype);
    SSWIN_CHECK(epilogue >= 0 && epilogue <= 3, "dense_forward: epilogue %d", epilogue);
    SSWIN_CHECK(transposed ? epilogue == EPI_NONE || epilogue == EPI_SCALE : epilogue != EPI_SCALE, "dense_forward: epilogue %d does not go with transposed = %d",
                epilogue, transposed);
    SSWIN_CHECK(epilogue < EPI_RESIDUAL || extra || N == 0, "dense_forward: the epilogue needs its second operand");
    if (N == 0) return 0;
    SSWIN_CHECK(x && w && y, "dense_forward: null pointer");
    SSWIN_CHECK(((uintptr_t)x | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)extra | (uintptr_t)y | (uintptr_t)slope) % 16 == 0,
                "dense_forward: pointers must be 16-byte aligned");
    const Epilogue ep = {bias, extra, y, slope};
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool down = transposed != 0;
#define DENSE_RUN(T, TB, TO) return pick_forward<T, TB, TO>(epilogue, down, x, N, K, w, P, ep, s)
    if (dtype == SSWIN_F32 && w_dtype == SSWIN_F32 && out_dtype == SSWIN_F32) DENSE_RUN(float, float, float);
    if (dtype == SSWIN_F16 && w_dtype == SSWIN_F16 && out_dtype == SSWIN_F16) DENSE_RUN(__half, __half, __half);
    if (dtype == SSWIN_BF16 && w_dtype == SSWIN_BF16 && out_dtype == SSWIN_BF16) DENSE_RUN(__hip_bfloat16, __hip_bfloat16, __hip_bfloat16);
    if (dtype == SSWIN_F16 && w_dtype == SSWIN_F32 && out_dtype == SSWIN_F16) DENSE_RUN(__half, float, __half);
    if (dtype == SSWIN_BF16 && w_dtype == SSWIN_F32 && out_dtype == SSWIN_BF16) DENSE_RUN(__hip_bfloat16, float, __hip_bfloat16);
    if (epilogue == EPI_RESIDUAL) {                                      // mixed precision: the residual stream stays fp32
        if (dtype == SSWIN_F16 && w_dtype == SSWIN_F32 && out_dtype == SSWIN_F32)
            return launch_forward<__half, float, float, EPI_RESIDUAL, false>(x, N, K, w, P, ep, s);
        if (dtype == SSWIN_BF16 && w_dtype == SSWIN_F32 && out_dtype == SSWIN_F32)
            return launch_forward<__hip_bfloat16, float, float, EPI_RESIDUAL, false>(x, N, K, w, P, ep, s);
    }
#undef DENSE_RUN
    return fail("dense_forward: tokens of type %d with weights of type %d and a result of type %d are not supported", dtype, w_dtype, out_dtype);
}

size_t sswin_dense_weight_grad_workspace_bytes(int dtype, int64_t N, int P, int K) {
    if (N <= 0 || !sswin_dense_supported(dtype, P, K)) return 0;
    const WgradPlan pl = wgrad_plan(dtype, N, P, K);
    return (size_t)pl.chunks * ((size_t)P * K + P) * sizeof(float);
}

int sswin_dense_weight_grad(int dtype, int out_dtype, const void* dy, const void* x, int64_t N, int P, int K, void* dw, void* db, void* ws, size_t ws_bytes,
                            void* stream) {
    SSWIN_CHECK(N > 0, "dense_weight_grad: bad sizes");
    SSWIN_CHECK(sswin_dense_supported(dtype, P, K), "dense_weight_grad: %d -> %d channels of type %d are not supported (multiples of 16)", K, P, dtype);
    SSWIN_CHECK(dy && x && dw && ws, "dense_weight_grad: null pointer");
    SSWIN_CHECK(((uintptr_t)dy | (uintptr_t)x | (uintptr_t)dw | (uintptr_t)db | (uintptr_t)ws) % 16 == 0, "dense_weight_grad: pointers must be 16-byte aligned");
    SSWIN_CHECK(ws_bytes >= sswin_dense_weight_grad_workspace_bytes(dtype, N, P, K), "dense_weight_grad: workspace too small");
    hipStream_t s = static_cast<hipStream_t>(stream);
    float* f = static_cast<float*>(ws);
    if (dtype == SSWIN_F32 && out_dtype == SSWIN_F32) return launch_wgrad<float, float>(dy, x, N, P, K, dw, db, f, s);
    if (dtype == SSWIN_F16 && out_dtype == SSWIN_F16) return launch_wgrad<__half, __half>(dy, x, N, P, K, dw, db, f, s);
    if (dtype == SSWIN_F16 && out_dtype == SSWIN_F32) return launch_wgrad<__half, float>(dy, x, N, P, K, dw, db, f, s);
    if (dtype == SSWIN_BF16 && out_dtype == SSWIN_BF16) return launch_wgrad<__hip_bfloat16, __hip_bfloat16>(dy, x, N, P, K, dw, db, f, s);
    if (dtype == SSWIN_BF16 && out_dtype == SSWIN_F32) return launch_wgrad<__hip_bfloat16, float>(dy, x, N, P, K, dw, db, f, s);
    return fail("dense_weight_grad: operands of type %d with a result of type %d are not supported", dtype, out_dtype);
}

}  // extern "C"
