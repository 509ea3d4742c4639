// Dense layers over all tokens (nn.Linear of sparse_swin/swin3d_base.py:606-610 and of the feed-forward part,
// :722-735), forward, input gradient and weight gradient, for fp32, fp16 and bf16 tokens, with what follows the
// product folded into its last step: bias, GELU and its derivative, the product with that derivative, the residual sum.
//
// Products run on the 16-bit matrix cores with fp32 accumulation.  fp32 operands are split exactly into three bf16
// pieces (x = h + m + l, split2 of dense_operand.hpp) and a product is the sum of the six piece products that
// weigh at least 2^-16 of the leading one; what is dropped is below 2^-23 of the product.  Infinities and NaN give what they give
// in plain fp32 (plain_products).
//
// (dense_pairs.hip: layers of at least 96 reduction channels, with a workspace, as two fp16 pieces.)
// dense_rows_kernel (fp32): a workgroup of WM wavefronts owns BM = 32 MT WM rows and 32 NT columns, 64 or 96.  Both operands pass through
// registers, where they are split, into LDS in matrix operand order, [row tile][plane][lane] pieces of 16 bytes, so that every
// operand read is one conflict-free 16-byte read per lane; 32 columns of the reduction at a time, the next 32 in flight
// meanwhile.  96 columns because every layer of a stage has a multiple of 48, 64 where that wastes no more of them.  The tile of the result goes back
// through LDS, so that bias, residual and result are touched in 16-byte pieces of whole row segments.
// dense16_rows_kernel (16 bit): tiles straight from memory to LDS.
// dense_small_kernel: few rows and many channels (the deep stages): 32 x 32 tiles, the wavefronts of a workgroup share
// the reduction instead of the rows, so that a few hundred rows still put a wavefront on every SIMD.
// dense_wgrad_kernel, dense16_wgrad_kernel: dW = dY^T X, db = column sums of dY: the reduction runs over the rows; fp32 operands
// are read as 8 rows x 2 columns per lane and turned in registers, 16-bit ones by the transposing LDS load.  Row chunks are
// added by a second kernel in a fixed order.
#include <math.h>

#include <algorithm>

#include "dense_epilogue.hpp"
#include "dense_operand.hpp"
#include "mfma_block.hpp"
#include "sswin_common.hpp"

namespace sswin {
namespace dense {

// ------------------------------------------------------------------------------------------
// Raw values of a unit on their way from memory to LDS.
// Along: 8 consecutive values of one row (reduction along the row).  Down: 8 rows x 2 columns (reduction down the rows).
// ------------------------------------------------------------------------------------------
template <typename T> struct Along {
    static constexpr bool WIDE = sizeof(T) == 4;
    u32x4 r[WIDE ? 2 : 1];
    __device__ __forceinline__ void load(const T* p) {
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

struct Down {
    uint32_t r[8][2];
    __device__ __forceinline__ void load(int e, const float* p) {
        r[e][0] = reinterpret_cast<const uint32_t*>(p)[0];
        r[e][1] = reinterpret_cast<const uint32_t*>(p)[1];
    }
    __device__ __forceinline__ void zero(int e) { r[e][0] = r[e][1] = 0; }
    // column c (0 or 1) of the pair
    __device__ __forceinline__ void planes(int c, u32x4 (&out)[3]) const {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = __builtin_bit_cast(float, r[e][c]);
        planes_of<float>(v, out);
    }
    __device__ __forceinline__ float sum(int c) const {
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) s += __builtin_bit_cast(float, r[e][c]);
        return s;
    }
};
template <typename T> __device__ __forceinline__ float half_of(uint32_t w, int c);
template <> __device__ __forceinline__ float half_of<__half>(uint32_t w, int c) {
    return __half2float(__ushort_as_half((unsigned short)(c ? w >> 16 : w & 0xffffu)));
}
template <> __device__ __forceinline__ float half_of<__hip_bfloat16>(uint32_t w, int c) {
    return __builtin_bit_cast(float, c ? w & 0xffff0000u : w << 16);
}

// position of (row, 8-value chunk) inside its 32-row operand block: the rows of a chunk are rotated by the chunk, so
// that lanes which hold the chunks of one row write to different banks
__device__ __forceinline__ int swz(int chunk) { return (chunk & 1) * 4 | (chunk & 2); }

// ------------------------------------------------------------------------------------------
// y [N, P] = last step of x [N, K] Wop, Wop [K, P] = W^T of W [P, K] (DOWN = false) or W [K, P] itself (DOWN = true)
// ------------------------------------------------------------------------------------------
template <int EPI, bool DOWN, int WM, int MT, int NT, int OCC>
__global__ __launch_bounds__(WM * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void dense_rows_kernel(
    const float* __restrict__ x, int64_t N, int K, const float* __restrict__ w, int P, int groups, Epilogue ep) {
    constexpr int PL = 3, BK = 32, KC = BK / 8;
    constexpr int BN = NT * 32, BM = WM * MT * 32, THREADS = WM * 64;
    constexpr int A_UNITS = BM * KC, UA = (A_UNITS + THREADS - 1) / THREADS;
    constexpr int B_UNITS = (DOWN ? BN / 2 : BN) * KC, UB = (B_UNITS + THREADS - 1) / THREADS;
    constexpr int A_LDS = BM / 32 * PL * 64, B_LDS = NT * PL * 64;       // 16-byte pieces of 16 columns
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    int cg;
    int64_t rb;
    block_of(groups, cg, rb);
    const int64_t row0 = rb * BM;
    const int col0 = cg * BN;

    // addresses: a uniform base that moves along the reduction plus 32-bit lane offsets formed once
    Along<float> ra[UA];
    typename std::conditional<DOWN, Down, Along<float>>::type rw[UB];
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
    const float* xb = x + row0 * K;
    // 32 columns from k0 on; where only 16 are left, the upper half repeats them
    auto request = [&](int k0) {
        const bool half_step = k0 + 16 == K;
#pragma unroll
        for (int i = 0; i < UA; ++i) {
            const int u = threadIdx.x + i * THREADS;
            if (A_UNITS % THREADS == 0 || u < A_UNITS) ra[i].load(xb + k0 + (oa[i] - (half_step ? (u % KC / 2) * 16 : 0)));
        }
#pragma unroll
        for (int i = 0; i < UB; ++i) {
            const int u = threadIdx.x + i * THREADS;
            if (B_UNITS % THREADS == 0 || u < B_UNITS) {
                if constexpr (DOWN) {
                    const uint32_t at = ow[i] - (half_step ? u / (BN / 2) / 2 * 16 * P : 0);
#pragma unroll
                    for (int e = 0; e < 8; ++e) rw[i].load(e, w + (int64_t)(k0 + e) * P + at);
                } else {
                    rw[i].load(w + k0 + (ow[i] - (half_step ? (u % KC / 2) * 16 : 0)));
                }
            }
        }
    };
    auto put = [&](u32x4* base, int tiles, int row, int c, const u32x4 (&p)[PL]) {
        u32x4* dst = base + (((c >> 1) * tiles + (row >> 5)) * PL) * 64 + (c & 1) * 32 + ((row & 31) ^ swz(c));
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
                    put(buf + 2 * A_LDS, NT, (u % (BN / 2)) * 2, u / (BN / 2), p);
                    rw[i].planes(1, p);
                    put(buf + 2 * A_LDS, NT, (u % (BN / 2)) * 2 + 1, u / (BN / 2), p);
                } else {
                    rw[i].planes(p);
                    put(buf + 2 * A_LDS, NT, u / KC, u % KC, p);
                }
            }
        }
    };

    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    // One buffer of 32 columns, whole 128-byte lines of x and w: in steps of 16 columns a line was fetched from L2 twice, once
    // per half, since the rows of three workgroups overflow L1 in between (219 000 rows 288 -> 96 and 384 -> 96, input gradients: 96 us
    // on average, with whole lines 87; 384 -> 96 with a residual 171 and 166; the traffic's own time is 72 and 95).
    request(0);
    for (int k0 = 0; k0 < K; k0 += BK) {
        if (k0) __syncthreads();                                         // the last step's operands have been read
        store(lds);
        if (k0 + BK < K) request(k0 + BK);
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (h && k0 + 16 == K) break;
            const int at = half * 32 + (l32 ^ swz(2 * h + half));
            u32x4 a[MT][PL], b[NT][PL];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int q = 0; q < PL; ++q) a[i][q] = lds[h * A_LDS + ((wave * MT + i) * PL + q) * 64 + at];
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < PL; ++q) b[j][q] = lds[2 * A_LDS + h * B_LDS + (j * PL + q) * 64 + at];
#pragma unroll
            for (int p = 0; p < Op<float>::NP; ++p)
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = Op<float>::mfma(a[i][Op<float>::PA[p]], b[j][Op<float>::PB[p]], acc[i][j]);
        }
    }
    __syncthreads();
    // the tile of the wavefront, 32 rows at a time, through its own part of LDS (pitch 100: rows start 4 banks apart)
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
        constexpr int PIECES = 32 * (BN / 4) / 64;
        f32x4 any = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) any[r & 3] += acc[i][j][r];
        if (__any(nan_among(any))) {
#pragma unroll 1
            for (int q = 0; q < PIECES; ++q) {
                const int e = q * 64 + lane, rr = e / (BN / 4), cc = (e % (BN / 4)) * 4;
                f32x4* v = reinterpret_cast<f32x4*>(mine + rr * PITCH + cc);
                if (r0 + rr < N && col0 + cc < P && nan_among(*v))
                    *v = plain_products(x + (r0 + rr) * K, 1, w + (DOWN ? col0 + cc : (int64_t)(col0 + cc) * K), DOWN ? P : 1, DOWN ? 1 : K, K);
            }
            __builtin_amdgcn_wave_barrier();
        }
        Second4<float, float, EPI> second[PIECES];
#pragma unroll
        for (int q = 0; q < PIECES; ++q) {
            const int e = q * 64 + lane, rr = e / (BN / 4), cc = (e % (BN / 4)) * 4;
            if (r0 + rr < N && col0 + cc < P) second[q].load(ep, r0 + rr, col0 + cc, P);
        }
#pragma unroll
        for (int q = 0; q < PIECES; ++q) {
            const int e = q * 64 + lane, rr = e / (BN / 4), cc = (e % (BN / 4)) * 4;
            const f32x4 v = *reinterpret_cast<const f32x4*>(mine + rr * PITCH + cc);
            if (r0 + rr < N && col0 + cc < P) finish4<float, float, EPI>(ep, r0 + rr, col0 + cc, P, v, second[q]);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// ------------------------------------------------------------------------------------------
// 16-bit operands: the same products with tiles that go from memory to LDS directly (no registers in between), the next
// block of the reduction in flight, and operands that lie across the reduction read through the transposing LDS load
// (ds_read_b64_tr_b16: a group of 16 lanes reads 4 rows x 16 columns and lane i receives column i).
//
// Tile layouts are the memory's own: [row][BK] for operands along the reduction, the pieces of a row exchanged;
// [row of the reduction][96] for operands down the reduction (192-byte rows: the four rows of a transposing read lie in
// different banks).  A wavefront waits for its own loads of the oldest block (vmcnt), one barrier makes the block
// complete, the next loads go into the buffer that was read one block ago.
//
// WM x WN wavefronts share the tile (32 MT rows x 96 columns each), KG = 2 groups of them the steps of a block.  What
// bounds it: at 96 channels the traffic of the result (219 000 rows 96 -> 288, 168 MB: 44 us, with operands through registers
// 57; its input gradient 33 and 43), at long reductions what passes from L2 into LDS, 14 TB/s over the chip (8119 rows
// 768 -> 3072: 57 us, through registers 73).
// ------------------------------------------------------------------------------------------
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;

// place of a 16-byte piece in its row of BK values: pieces are exchanged by the row's number, so that the lanes of a read
// (consecutive rows, the same piece) lie in different banks
template <int BK> __device__ __forceinline__ int swapped(int row, int piece) {
    static_assert(BK == 32 || BK == 64, "four or eight pieces a row");
    return BK == 32 ? piece ^ (((row >> 1) ^ (row >> 3)) & 3) : piece ^ (row & 7);
}
// operand of 32 rows x 16 reduction slots from a tile whose rows run along the reduction
template <typename T, int BK>
__device__ __forceinline__ u32x4 along_operand(const T* tile, int row0, int ks) {
    const int row = row0 + (threadIdx.x & 31);
    return *reinterpret_cast<const u32x4*>(tile + row * BK + swapped<BK>(row, ks * 2 + ((threadIdx.x & 63) >> 5)) * 8);
}
// the same from a tile whose rows run across it ([reduction][96])
template <typename T>
__device__ __forceinline__ u32x4 down_operand(const T* tile, int col, int ks) {
    const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
    const T* p = tile + (ks * 16 + (g >> 1) * 8 + (i >> 2)) * 96 + col + (g & 1) * 16 + (i & 3) * 4;
    union {
        s16x4_t h[2];
        u32x4 v;
    } o;
    o.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
    o.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * 96));
    return o.v;
}

template <typename T, typename TO, int EPI, bool DOWN, int BK, int WM, int WN, int KG, int MT, int STAGES, int OCC>
__global__ __launch_bounds__(WM * WN * KG * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void dense16_rows_kernel(
    const T* __restrict__ x, int64_t N, int K, const T* __restrict__ w, int P, int groups, int ksplit, float* __restrict__ part, Epilogue ep) {
    constexpr int PR = BK / 8, NT = 3, BN = 96 * WN, BM = WM * MT * 32, THREADS = WM * WN * KG * 64;
    constexpr int A_PIECES = BM * PR, B_PIECES = BN * PR, UA = (A_PIECES + THREADS - 1) / THREADS, UB = (B_PIECES + THREADS - 1) / THREADS;
    static_assert(A_PIECES % 64 == 0 && B_PIECES % 64 == 0 && BK % (16 * KG) == 0, "whole wavefronts of pieces");
    constexpr int BUF = (A_PIECES + B_PIECES) * 8;                       // values
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
    T* const tiles = reinterpret_cast<T*>(lds);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int wk = wave / (WM * WN), wm = wave % (WM * WN) / WN, wn = wave % WN;
    int cg;
    int64_t rb;
    block_of(groups * ksplit, cg, rb);
    const int part_no = cg / groups;                                     // share of the reduction
    cg %= groups;
    const int64_t row0 = rb * BM;
    const int col0 = cg * BN;
    const int all = (K + BK - 1) / BK, k_first = all * part_no / ksplit, nk = all * (part_no + 1) / ksplit - k_first;
    const int last = (int)(N - 1 - row0 < BM - 1 ? N - 1 - row0 : BM - 1);   // rows past the end repeat the last one
    // this lane's pieces: row and first value of a piece of X; row (of the output, or of the reduction) and first value of Wop
    const T* pa[UA];
    const T* pb[UB];
    auto a_k = [](int u) { return swapped<BK>(u / PR, u % PR) * 8; };
    auto b_k = [](int u) { return DOWN ? u % (BK * 12) / 12 : swapped<BK>(u / PR, u % PR) * 8; };
#pragma unroll
    for (int i = 0; i < UA; ++i) {
        const int u = i * THREADS + threadIdx.x;
        pa[i] = x + (row0 + min(u / PR, last)) * K + k_first * BK + a_k(u);
    }
#pragma unroll
    for (int i = 0; i < UB; ++i) {
        const int u = i * THREADS + threadIdx.x;
        if (DOWN) pb[i] = w + (int64_t)(k_first * BK + b_k(u)) * P + min(col0 + u / (BK * 12) * 96 + (u % 12) * 8, P - 8);
        else pb[i] = w + (int64_t)min(col0 + u / PR, P - 1) * K + k_first * BK + b_k(u);
    }
    const int64_t step_b = DOWN ? (int64_t)BK * P : BK;
    const uint32_t base = lds_address(tiles);
    auto request = [&](int kb) {
        const uint32_t buf = base + (uint32_t)(kb % STAGES) * BUF * 2;
        const int k0 = (k_first + kb) * BK;
        const bool ragged = k0 + BK > K;                                 // then the last piece or row inside; cleared below
#pragma unroll
        for (int i = 0; i < UA; ++i)
            if (i * THREADS + wave * 64 < A_PIECES) {                    // uniform in the wavefront
                const int over = ragged ? max(k0 + a_k(i * THREADS + threadIdx.x) - (K - 8), 0) : 0;
                copy_to_lds(pa[i] - over, buf + (uint32_t)(i * THREADS + wave * 64) * 16);
                pa[i] += BK;
            }
#pragma unroll
        for (int i = 0; i < UB; ++i)
            if (i * THREADS + wave * 64 < B_PIECES) {
                const int over = ragged ? max(k0 + b_k(i * THREADS + threadIdx.x) - (K - (DOWN ? 1 : 8)), 0) : 0;
                copy_to_lds(pb[i] - (DOWN ? (int64_t)over * P : over), buf + (uint32_t)(A_PIECES + i * THREADS + wave * 64) * 16);
                pb[i] += step_b;
            }
    };
    // a wavefront's loads per block, for the counter of outstanding loads: all wavefronts wait for the smallest number that is safe
    constexpr int FEWEST = A_PIECES / THREADS + B_PIECES / THREADS;

    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < STAGES - 1; ++p)
        if (p < nk) request(p);
    for (int kb = 0; kb < nk; ++kb) {
        if (kb + STAGES - 1 <= nk) wait_copies<FEWEST * (STAGES - 2)>();
        else wait_copies<0>();
        block_barrier();
        if (kb + STAGES - 1 < nk) request(kb + STAGES - 1);
        T* ta = tiles + (kb % STAGES) * BUF;
        T* tb = ta + A_PIECES * 8;
        const int left = K - (k_first + kb) * BK;
        if (left < BK) {
            for (int u = threadIdx.x; u < A_PIECES; u += THREADS)
                if (a_k(u) >= left) reinterpret_cast<u32x4*>(ta)[u] = u32x4{0, 0, 0, 0};
            for (int u = threadIdx.x; u < B_PIECES; u += THREADS)
                if (b_k(u) >= left) reinterpret_cast<u32x4*>(tb)[u] = u32x4{0, 0, 0, 0};
            block_barrier();
        }
#pragma unroll
        for (int q = 0; q < BK / 16 / KG; ++q) {
            const int ks = wk * (BK / 16 / KG) + q;
            u32x4 a[MT], b[NT];
#pragma unroll
            for (int i = 0; i < MT; ++i) a[i] = along_operand<T, BK>(ta, (wm * MT + i) * 32, ks);
#pragma unroll
            for (int j = 0; j < NT; ++j) b[j] = DOWN ? down_operand(tb + wn * BK * 96, j * 32, ks) : along_operand<T, BK>(tb, wn * 96 + j * 32, ks);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = Op<T>::mfma(a[i], b[j], acc[i][j]);
        }
    }
    block_barrier();
    if constexpr (KG == 2) {                                             // the two halves of each block's steps
        float* other = reinterpret_cast<float*>(lds) + (wave % (WM * WN)) * MT * NT * 16 * 64;
        if (wk == 1) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) other[((i * NT + j) * 16 + r) * 64 + lane] = acc[i][j][r];
        }
        block_barrier();
        if (wk == 0) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] += other[((i * NT + j) * 16 + r) * 64 + lane];
        }
        block_barrier();
        if (wk == 1) return;
    }
    // Through LDS, 16 rows x 96 columns of a wavefront at a time, so that every lane holds eight neighbouring columns and a row
    // leaves in one run of 192 bytes (32 columns at a time, runs of 64 bytes: 450 000 rows 96 -> 288 bf16 138 us, now 115;
    // 219 000 rows 96 -> 96 with a residual 31 and 25; 192 -> 48 times a factor, fp16, 59 and 41)
    constexpr int PITCH = 100, PIECES = 16 * 12 / 64;
    float* mine = reinterpret_cast<float*>(lds) + wave * 16 * PITCH;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int64_t r0 = row0 + (wm * MT + i) * 32 + h * 16;
            const int c0 = col0 + wn * 96;
            Second8<T, TO, EPI> second[PIECES];
            if (!part)
#pragma unroll
                for (int q = 0; q < PIECES; ++q) {
                    const int e = q * 64 + lane, rr = e / 12, cc = e % 12 * 8;
                    if (r0 + rr < N && c0 + cc < P) second[q].load(ep, r0 + rr, c0 + cc, P);
                }
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 8; ++r) mine[acc_row(r, half) * PITCH + j * 32 + l32] = acc[i][j][h * 8 + r];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < PIECES; ++q) {
                const int e = q * 64 + lane, rr = e / 12, cc = e % 12 * 8;
                const f32x4 v[2] = {*reinterpret_cast<const f32x4*>(mine + rr * PITCH + cc), *reinterpret_cast<const f32x4*>(mine + rr * PITCH + cc + 4)};
                const int64_t row = r0 + rr;
                const int col = c0 + cc;
                if (row < N && col < P) {
                    if (part) {
                        f32x4* at = reinterpret_cast<f32x4*>(part + ((int64_t)part_no * N + row) * P + col);
                        at[0] = v[0];
                        at[1] = v[1];
                    } else {
                        finish8<T, TO, EPI>(ep, row, col, P, v, second[q]);
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
}

// the shares of the reduction added in order, then the last step
template <typename T, typename TO, int EPI>
__global__ __launch_bounds__(256) void dense_parts_kernel(const float* __restrict__ part, int64_t N, int P, int parts, Epilogue ep) {
    const int64_t quads = N * (P / 4), i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= quads) return;
    const int64_t row = i / (P / 4);
    const int col = (int)(i % (P / 4)) * 4;
    Second4<T, TO, EPI> second;
    second.load(ep, row, col, P);
    f32x4 v = *reinterpret_cast<const f32x4*>(part + i * 4);
    for (int p = 1; p < parts; ++p) v += *reinterpret_cast<const f32x4*>(part + (int64_t)p * N * P + i * 4);
    finish4<T, TO, EPI>(ep, row, col, P, v, second);
}

// dW [P, K] = dY^T X for one chunk of rows; WM x WN wavefronts of (32 MT) x 96 each, BM = 32 MT WM columns of dY (a multiple of
// 96), BN = 96 WN columns of X
// (219 000 rows 96 -> 288, 168 MB: 39 us; 384 -> 96 45; the traffic's own time at copy rate is 33 and 41)
template <typename T, int WM, int WN, int MT, int STAGES, int OCC>
__global__ __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void dense16_wgrad_kernel(
    const T* __restrict__ dy, const T* __restrict__ x, int64_t N, int P, int K, int tiles_p, int tiles_k, int64_t rows_per_chunk, float* __restrict__ part_w,
    float* __restrict__ part_b) {
    constexpr int BK = 32, NT = 3, BM = WM * MT * 32, BN = WN * 96, THREADS = WM * WN * 64;
    static_assert(BM % 96 == 0, "sub-tiles of 96 columns");
    constexpr int SUB = BK * 12;                                         // pieces of a sub-tile of 96 columns
    constexpr int PIECES = (BM / 96 + WN) * SUB, U = PIECES / THREADS, BUF = PIECES * 8;
    static_assert(PIECES % THREADS == 0, "whole rounds of pieces");
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
    T* const tiles = reinterpret_cast<T*>(lds);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int wm = wave / WN, wn = wave % WN;
    int tile;
    int64_t chunk;
    block_of(tiles_p * tiles_k, tile, chunk);
    const int p0 = (tile / tiles_k) * BM, k0 = (tile % tiles_k) * BN;
    const int64_t begin = chunk * rows_per_chunk, end = begin + rows_per_chunk < N ? begin + rows_per_chunk : N;
    const int nk = (int)((end - begin + BK - 1) / BK);
    const bool sums_here = part_b && k0 == 0 && wn == 0;
    // piece u: sub-tile u / SUB (those of dY first), row (u % SUB) / 12, 8 columns u % 12
    auto source = [&](int u, int64_t n0) -> const T* {
        const int sub = u / SUB, r = u % SUB / 12, c = u % 12 * 8;
        const int64_t n = n0 + r < end ? n0 + r : end - 1;               // rows past the end are cleared below
        if (sub < BM / 96) return dy + n * P + min(p0 + sub * 96 + c, P - 8);
        return x + n * K + min(k0 + (sub - BM / 96) * 96 + c, K - 8);
    };
    const T* p[U];
    int64_t step[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
        const int u = i * THREADS + threadIdx.x;
        p[i] = source(u, begin);
        step[i] = (int64_t)BK * (u / SUB < BM / 96 ? P : K);
    }
    const uint32_t base = lds_address(tiles);
    auto request = [&](int kb) {
        const uint32_t buf = base + (uint32_t)(kb % STAGES) * BUF * 2;
        const bool ragged = begin + (int64_t)(kb + 1) * BK > end;
#pragma unroll
        for (int i = 0; i < U; ++i) {
            copy_to_lds(ragged ? source(i * THREADS + threadIdx.x, begin + (int64_t)kb * BK) : p[i], buf + (uint32_t)(i * THREADS + wave * 64) * 16);
            p[i] += step[i];
        }
    };
    f32x16 acc[MT][NT];
    float bs[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        bs[i] = 0.f;
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int q = 0; q < STAGES - 1; ++q)
        if (q < nk) request(q);
    for (int kb = 0; kb < nk; ++kb) {
        if (kb + STAGES - 1 <= nk) wait_copies<U * (STAGES - 2)>();
        else wait_copies<0>();
        block_barrier();
        if (kb + STAGES - 1 < nk) request(kb + STAGES - 1);
        T* t = tiles + (kb % STAGES) * BUF;
        const int left = (int)(end - begin - (int64_t)kb * BK);
        if (left < BK) {                                                 // the last block of the rows: zero past the end
            for (int q = threadIdx.x; q < PIECES; q += THREADS)
                if (q % SUB / 12 >= left) reinterpret_cast<u32x4*>(t)[q] = u32x4{0, 0, 0, 0};
            block_barrier();
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            u32x4 a[MT], b[NT];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int col = (wm * MT + i) * 32;
                a[i] = down_operand(t + col / 96 * SUB * 8, col % 96, ks);
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) b[j] = down_operand(t + (BM / 96 + wn) * SUB * 8, j * 32, ks);
            if (sums_here) {
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    float s = 0.f;
#pragma unroll
                    for (int e = 0; e < 4; ++e) s += half_of<T>(a[i][e], 0) + half_of<T>(a[i][e], 1);
                    bs[i] += s;
                }
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = Op<T>::mfma(a[i], b[j], acc[i][j]);
        }
    }
    float* pw = part_w + chunk * (int64_t)P * K;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int pp = p0 + (wm * MT + i) * 32 + acc_row(r, half), kk = k0 + wn * 96 + j * 32 + l32;
                if (pp < P && kk < K) pw[(int64_t)pp * K + kk] = acc[i][j][r];
            }
        if (sums_here) {
            const float s = bs[i] + __shfl_xor(bs[i], 32, 64);           // the two halves of the reduction slots
            const int pp = p0 + (wm * MT + i) * 32 + l32;
            if (half == 0 && pp < P) part_b[chunk * P + pp] = s;
        }
    }
}

// ------------------------------------------------------------------------------------------
// The same for few rows: a workgroup owns a 32 x 32 tile, its 8 wavefronts take every 8th 16-wide step of the reduction
// and add their tiles through LDS in a fixed order.
// ------------------------------------------------------------------------------------------
constexpr int SMALL_WAVES = 8;
struct SmallLds {
    __attribute__((aligned(16))) float sums[SMALL_WAVES][32 * 36];
    float colsum[SMALL_WAVES][64];
};
template <typename T, typename TO, int EPI, bool DOWN>
__device__ __forceinline__ void small_tile(int block, const T* __restrict__ x, int64_t N, int K, const T* __restrict__ w, int P, int groups,
                                           const Epilogue& ep, float (&sums)[SMALL_WAVES][32 * 36]) {
    constexpr int PL = Op<T>::PL;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int64_t row0 = (int64_t)(block / groups) * 32;
    const int col0 = block % groups * 32, steps = K / 16;
    const int64_t row = row0 + l32 < N ? row0 + l32 : N - 1;
    const int col = min(col0 + l32, P - 1);
    const T* xp = x + row * K + half * 8;
    f32x16 acc = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    constexpr int AHEAD = 3;                                             // steps of a wavefront in flight
    Along<T> ra[AHEAD];
    Along<T> rb[DOWN ? 1 : AHEAD];
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
        const bool in = row0 + rr < N && col0 + cc < P;
        Second4<T, TO, EPI> second;
        if (in) second.load(ep, row0 + rr, col0 + cc, P);
        f32x4 v = *reinterpret_cast<const f32x4*>(&sums[0][rr * 36 + cc]);
#pragma unroll
        for (int q = 1; q < SMALL_WAVES; ++q) v += *reinterpret_cast<const f32x4*>(&sums[q][rr * 36 + cc]);
        if constexpr (PL == 3)
            if (__builtin_expect(in && nan_among(v), 0))
                v = plain_products(x + (row0 + rr) * K, 1, w + (DOWN ? col0 + cc : (int64_t)(col0 + cc) * K), DOWN ? P : 1, DOWN ? 1 : K, K);
        if (in) finish4<T, TO, EPI>(ep, row0 + rr, col0 + cc, P, v, second);
    }
}
template <typename T, typename TO, int EPI, bool DOWN>
__global__ __launch_bounds__(SMALL_WAVES * 64) void dense_small_kernel(const T* __restrict__ x, int64_t N, int K, const T* __restrict__ w, int P,
                                                                    int groups, Epilogue ep) {
    __shared__ SmallLds lds;
    small_tile<T, TO, EPI, DOWN>((int)blockIdx.x, x, N, K, w, P, groups, ep, lds.sums);
}

// ------------------------------------------------------------------------------------------
// dW [P, K] = dY^T X, db [P] = column sums of dY.  A workgroup owns BM x BN of dW for one chunk of rows; WK groups of its wavefronts
// take 16 rows of a step each, and their sums are added through LDS at the end.
// Bound by the splitting into planes (120 vector instructions a wavefront and step) next to the products.  Therefore:
//   12 wavefronts a compute unit in one workgroup, which also writes one partial sum (two workgroups of 6 do not fit next to each
//   other: 219 000 rows 384 -> 96 150 us, one of 12 with two row groups 121, four wavefronts of 64 x 96 before 155);
//   one unit of 8 x 2 values a lane at most, and the next step's splitting between this step's products, without a branch (with two
//   units on some wavefronts every one splits twice: 96 -> 384 rows 207 us, now 118);
//   rows requested two steps ahead, with waits that count (the loop waited for everything it had requested: a branch stood
//   between).
// ------------------------------------------------------------------------------------------
template <int WM, int WN, int WK, int MT, int NT, int OCC>
__global__ __launch_bounds__(WM * WN * WK * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void dense_wgrad_kernel(
    const float* __restrict__ dy, const float* __restrict__ x, int64_t N, int P, int K, int tiles_p, int tiles_k, int64_t rows_per_chunk,
    float* __restrict__ part_w, float* __restrict__ part_b) {
    constexpr int PL = 3, BK = 16 * WK, WAVES = WM * WN;                 // waves of a row part
    constexpr int BM = WM * MT * 32, BN = WN * NT * 32, THREADS = WK * WAVES * 64;
    // A unit is 8 rows of two columns; a wavefront takes 64 units of dY or 64 of X
    constexpr int A_UNITS = BM, B_UNITS = BN, A_WAVES = (A_UNITS + 63) / 64, B_WAVES = (B_UNITS + 63) / 64;
    static_assert(A_WAVES + B_WAVES <= WAVES, "a unit for every lane at most");
    constexpr int A_LDS = BM / 32 * PL * 64, B_LDS = BN / 32 * PL * 64, BUF = A_LDS + B_LDS;
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];          // [buffer 2][row part][dY, X][32 columns][plane][lane]
    const int id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = id % WAVES, part = id / WAVES, lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int wm = wave / WN, wn = wave % WN;
    int tile;
    int64_t chunk;
    block_of(tiles_p * tiles_k, tile, chunk);
    const int p0 = (tile / tiles_k) * BM, k0 = (tile % tiles_k) * BN;
    u32x4* planes = lds + part * BUF;
    const int64_t begin = chunk * rows_per_chunk, end = begin + rows_per_chunk < N ? begin + rows_per_chunk : N;

    // Lanes without a unit of their own read, split and store the last one again: no branch, so that the waits can count the loads and
    // the splitting can go between the products
    const bool of_a = wave < A_WAVES;
    const int own = (of_a ? wave : min(wave - A_WAVES, B_WAVES - 1)) * 64 + lane, unit = min(own, (of_a ? A_UNITS : B_UNITS) - 1);
    const int pairs = of_a ? BM / 2 : BN / 2, eight = unit / pairs, column = unit % pairs * 2, first_row = part * 16 + eight * 8;
    const int pitch = of_a ? P : K;
    const float* rows = of_a ? dy : x;
    const uint32_t from = (uint32_t)(first_row * pitch + (of_a ? min(p0 + column, P - 2) : min(k0 + column, K - 2)));
    u32x4* to = planes + (of_a ? 0 : A_LDS) + (column >> 5) * PL * 64 + eight * 32 + (column & 31);

    Down raw[2];                                                         // of the next two steps
    float bs[2] = {0.f, 0.f};
    auto request = [&](int slot, int64_t n0) {                           // a step of whole rows
#pragma unroll
        for (int e = 0; e < 8; ++e) raw[slot].load(e, rows + (n0 + e) * pitch + from);
    };
    auto request_end = [&](int slot, int64_t n0) {                       // zeros past the last row
        const int64_t left = end - n0 - first_row;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (e < left) raw[slot].load(e, rows + (n0 + e) * pitch + from);
            else raw[slot].zero(e);
        }
    };
    auto store = [&](int slot) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 p[PL];
            raw[slot].planes(h, p);
            bs[h] += raw[slot].sum(h);
#pragma unroll
            for (int q = 0; q < PL; ++q) to[slot * WK * BUF + h + q * 64] = p[q];
        }
    };
    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const int nk = (int)((end - begin + BK - 1) / BK), whole = (int)((end - begin) / BK);
    request_end(0, begin);
    if (nk > 1) request_end(1, begin + BK);
    store(0);
    if (nk > 2) request_end(0, begin + 2 * BK);
    auto products = [&](int slot) {
        const u32x4* buf = planes + slot * WK * BUF;
        u32x4 a[MT][PL];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < PL; ++q) a[i][q] = buf[((wm * MT + i) * PL + q) * 64 + lane];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            u32x4 b[PL];
#pragma unroll
            for (int q = 0; q < PL; ++q) b[q] = buf[A_LDS + ((wn * NT + j) * PL + q) * 64 + lane];
#pragma unroll
            for (int p = 0; p < Op<float>::NP; ++p)
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[i][j] = Op<float>::mfma(a[i][Op<float>::PA[p]], b[Op<float>::PB[p]], acc[i][j]);
        }
    };
    // Step kb multiplies its planes and splits the rows of kb + 1, requested two steps before; those of kb + 3 are requested then
    int kb = 0;
    constexpr int MFMAS = Op<float>::NP * MT * NT;
    for (; kb + 4 < whole; kb += 2) {
#pragma unroll
        for (int slot = 0; slot < 2; ++slot) {
            __syncthreads();
            products(slot);
            store(slot ^ 1);
            request(slot ^ 1, begin + (int64_t)(kb + slot + 3) * BK);
#pragma unroll
            for (int g = 0; g < MFMAS; ++g) {                            // the splitting between the products
                if (g == 0) __builtin_amdgcn_sched_group_barrier(0x100, (MT + 1) * PL, 0);
                if (g % (Op<float>::NP * MT) == 1 && g / (Op<float>::NP * MT) + 1 < NT) __builtin_amdgcn_sched_group_barrier(0x100, PL, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, (120 + MFMAS - 1) / MFMAS, 0);
                if (g >= MFMAS - 6) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    for (; kb < nk; kb += 2) {
#pragma unroll
        for (int slot = 0; slot < 2; ++slot) {
            if (kb + slot >= nk) break;
            __syncthreads();
            products(slot);
            if (kb + slot + 1 < nk) store(slot ^ 1);
            if (kb + slot + 3 < nk) request_end(slot ^ 1, begin + (int64_t)(kb + slot + 3) * BK);
        }
    }
#pragma unroll
    for (int q = 1; q < WK; ++q) {                                       // the sums of the other row parts, in order, onto those of part 0
        float* red = reinterpret_cast<float*>(lds) + wave * 64 + lane;
        __syncthreads();
        if (part == q) {
#pragma unroll
            for (int e = 0; e < MT * NT * 16; ++e) red[e * WAVES * 64] = acc[e / (NT * 16)][e / 16 % NT][e & 15];
        }
        __syncthreads();
        if (part == 0) {
#pragma unroll
            for (int e = 0; e < MT * NT * 16; ++e) acc[e / (NT * 16)][e / 16 % NT][e & 15] += red[e * WAVES * 64];
        }
    }
    if (part == 0) {
        float* pw = part_w + chunk * (int64_t)P * K;
        f32x4 any = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int p = p0 + (wm * MT + i) * 32 + acc_row(r, half), k = k0 + (wn * NT + j) * 32 + l32;
                    if (p < P && k < K) pw[(int64_t)p * K + k] = acc[i][j][r];
                    any[r & 3] += acc[i][j][r];
                }
        if (__builtin_expect(nan_among(any), 0)) {                              // those of this lane that are NaN, read back where they were stored
#pragma unroll 1
            for (int e = 0; e < MT * NT * 16; ++e) {
                const int p = p0 + (wm * MT + e / (NT * 16)) * 32 + acc_row(e & 15, half), k = k0 + (wn * NT + e / 16 % NT) * 32 + l32;
                if (p >= P || k >= K) continue;
                const float v = pw[(int64_t)p * K + k];
                if (v != v) pw[(int64_t)p * K + k] = plain_products(dy + begin * P + p, P, x + begin * K + k, K, 0, end - begin)[0];
            }
        }
    }
    if (part_b && k0 == 0) {
        // unit u of dY holds 8 rows u / (BM / 2) of its column pair: those of a pair are added in order
        __syncthreads();
        float* red = reinterpret_cast<float*>(lds);
        if (of_a && own == unit) red[(part * A_UNITS + unit) * 2] = bs[0], red[(part * A_UNITS + unit) * 2 + 1] = bs[1];
        __syncthreads();
        for (int c = threadIdx.x; c < BM; c += THREADS) {
            float s = 0.f;
#pragma unroll
            for (int q = 0; q < 2 * WK; ++q) s += red[(q * (BM / 2) + c / 2) * 2 + (c & 1)];
            if (p0 + c < P) part_b[chunk * P + p0 + c] = s;
        }
    }
}

// The same for few rows: a workgroup owns a 32 x 32 tile of dW, its 8 wavefronts take every 8th step of 16 rows and add
// their tiles through LDS in a fixed order, so that the result leaves in one launch.
template <typename T, typename TO>
__device__ __forceinline__ void wgrad_small_tile(int block, const T* __restrict__ dy, const T* __restrict__ x, int64_t N, int P, int K, int tiles_k,
                                                 TO* __restrict__ dw, TO* __restrict__ db, SmallLds& lds) {
    constexpr int PL = Op<T>::PL, AHEAD = 2;
    auto& sums = lds.sums;
    auto& colsum = lds.colsum;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    const int p0 = block / tiles_k * 32, k0 = block % tiles_k * 32;
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
            if constexpr (PL == 3)
                if (__builtin_expect(nan_among(v), 0)) v = plain_products(dy + p0 + rr, P, x + k0 + cc, K, 1, N);
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
template <typename T, typename TO>
__global__ __launch_bounds__(SMALL_WAVES * 64) void dense_wgrad_small_kernel(const T* __restrict__ dy, const T* __restrict__ x, int64_t N, int P, int K,
                                                                             int tiles_k, TO* __restrict__ dw, TO* __restrict__ db) {
    __shared__ SmallLds lds;
    wgrad_small_tile<T, TO>((int)blockIdx.x, dy, x, N, P, K, tiles_k, dw, db, lds);
}

// The whole backward of a layer on few rows: the input gradient's tiles, then the weight gradient's, which read the same dY and
// do not depend on them.  Latency bounds both; as two launches they run one after the other (500 rows fp32, 384 -> 1152 and
// 384 -> 384 on average: 18 us in two launches, 13 in one; 1536 -> 384 19 to 21 either way, bound by what passes from L2).
template <typename T, typename TO, int EPI>
__global__ __launch_bounds__(SMALL_WAVES * 64) void dense_backward_small_kernel(const T* __restrict__ dy, const T* __restrict__ x, const T* __restrict__ w,
                                                                                int64_t N, int P, int K, int dx_tiles, int tiles_k, Epilogue ep,
                                                                                TO* __restrict__ dw, TO* __restrict__ db) {
    __shared__ SmallLds lds;
    if ((int)blockIdx.x < dx_tiles) small_tile<T, T, EPI, true>((int)blockIdx.x, dy, N, P, w, K, tiles_k, ep, lds.sums);
    else wgrad_small_tile<T, TO>((int)blockIdx.x - dx_tiles, dy, x, N, P, K, tiles_k, dw, db, lds);
}

// out[e] = sum over chunks of part[chunk][e] for the weights and the bias behind each other; a block takes 4 EL outputs,
// CL = 256 / EL threads share four of them, each adds every CL-th chunk in order, the CL sums in a fixed tree.
// EL = 16; 4 from 256 chunks on, where small layers leave the chip idle and the sums one after the other take the time
// (1024 chunks of 144 x 48 and 48 x 48: 16.8 us on average, with 4 6.8), and for small fp32 layers from 150 (with the sums of 235
// chunks 144 x 48 21.4 -> 18.9 us and 2 % less rounding, 250 of 96 x 144 30.4 -> 29.1; 192 x 192 and 96 x 384 lose 4 us); 64 up to 16 chunks, where most of 16 threads have none
// (weight gradients of 2000 and 8119 rows 768 -> 2304: 35.5 -> 24.7 us and 73.0 -> 68.6)
template <typename TO, int EL>
__global__ __launch_bounds__(256) void dense_wgrad_sum_kernel(const float* __restrict__ part_w, const float* __restrict__ part_b, int chunks,
                                                              int64_t PK, int P, TO* __restrict__ dw, TO* __restrict__ db) {
    constexpr int CL = 256 / EL;
    __shared__ f32x4 sums[CL][EL + 1];
    const int el = threadIdx.x % EL, cl = threadIdx.x / EL;
    const int64_t e = ((int64_t)blockIdx.x * EL + el) * 4;
    const bool weight = e < PK, valid = weight || (db && e - PK < P);
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    if (valid) {
        const float* src = weight ? part_w + e : part_b + (e - PK);
        const int64_t pitch = weight ? PK : P;
        for (int c = cl; c < chunks; c += CL) sum += *reinterpret_cast<const f32x4*>(src + c * pitch);
    }
    sums[cl][el] = sum;
    __syncthreads();
#pragma unroll
    for (int w = CL / 2; w >= 1; w >>= 1) {
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
template <typename F> static int allow_lds(F* kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        SSWIN_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    return 0;
}

template <typename T, typename TO, int EPI>
static int launch_parts(const float* part, int64_t N, int P, int parts, const Epilogue& ep, hipStream_t s) {
    const int64_t blocks = (N * (P / 4) + 255) / 256;
    SSWIN_CHECK(blocks < (1ll << 31), "dense: too many rows");
    hipLaunchKernelGGL((dense_parts_kernel<T, TO, EPI>), dim3((unsigned)blocks), dim3(256), 0, s, part, N, P, parts, ep);
    return launch_ok("dense, parts");
}

template <int EPI, bool DOWN, int WM, int MT, int NT, int OCC>
static int launch_rows(const float* x, int64_t N, int K, const float* w, int P, const Epilogue& ep, hipStream_t s) {
    constexpr int BM = WM * MT * 32;
    constexpr size_t tiles = 2 * (size_t)(BM / 32 + NT) * 3 * 64 * 16, out = (size_t)WM * 32 * (NT * 32 + 4) * 4;
    constexpr size_t bytes = tiles > out ? tiles : out;
    auto* k = dense_rows_kernel<EPI, DOWN, WM, MT, NT, OCC>;
    static const int configured = allow_lds(k, bytes);
    if (configured) return configured;
    const int groups = (P + NT * 32 - 1) / (NT * 32);
    const int64_t blocks = (N + BM - 1) / BM * groups;
    SSWIN_CHECK(blocks < (1ll << 31), "dense: too many rows");
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(WM * 64), bytes, s, x, N, K, w, P, groups, ep);
    return launch_ok("dense");
}

template <typename T, typename TO, int EPI, bool DOWN, int BK, int WM, int WN, int KG, int MT, int STAGES, int OCC>
static int launch_rows16(const T* x, int64_t N, int K, const T* w, int P, int ksplit, float* ws, const Epilogue& ep, hipStream_t s) {
    constexpr int BM = WM * MT * 32, BN = WN * 96;
    constexpr size_t tiles = STAGES * (size_t)(BM + BN) * BK * 2, out = (size_t)WM * WN * (KG == 2 ? MT * 96 : 50) * 32 * 4;
    constexpr size_t bytes = tiles > out ? tiles : out;
    auto* k = dense16_rows_kernel<T, TO, EPI, DOWN, BK, WM, WN, KG, MT, STAGES, OCC>;
    static const int configured = allow_lds(k, bytes);
    if (configured) return configured;
    const int groups = (P + BN - 1) / BN;
    const int64_t blocks = (N + BM - 1) / BM * groups * ksplit;
    SSWIN_CHECK(blocks < (1ll << 31), "dense: too many rows");
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(WM * WN * KG * 64), bytes, s, x, N, K, w, P, groups, ksplit, ksplit > 1 ? ws : nullptr, ep);
    if (int rc = launch_ok("dense, 16 bit")) return rc;
    return ksplit > 1 ? launch_parts<T, TO, EPI>(ws, N, P, ksplit, ep, s) : 0;
}

// How a product is cut.
//   few rows: 32 x 32 tiles while the workgroups of the larger tiles would leave most of the chip idle.  fp32: below 150 tiles of
//     128 x 96.  16 bit: see few_line.
//   ksplit (16 bit): shares of the reduction, each at least 576 long, while the tiles alone do not fill the chip: 1364 rows
//     3072 -> 768 (88 tiles) 36 us with one share, 24 with two, 23 with four; 2729 rows (176 tiles) 37, 33 and 36.
struct Cut {
    bool few;
    int ksplit;
};
constexpr int64_t FEW_MOST = 50000;
static Cut cut_of(int dtype, int64_t N, int K, int P, int64_t line = FEW_MOST) {
    const int64_t tiles = (N + 127) / 128 * ((P + 95) / 96);
    if (dtype == SSWIN_F32) return {tiles < 150, 1};
    if (tiles * K <= line) return {true, 1};
    const int64_t shares = std::min<int64_t>({4, 400 / tiles, K / 576});
    return {false, (int)std::max<int64_t>(shares, 1)};
}
bool few_rows(int dtype, int64_t N, int K, int P) { return cut_of(dtype, N, K, P).few; }

// 16 bit: tiles x K up to which few rows are ahead.  Their time grows with it, that of the larger tiles starts at 6 us with the input
// gradient, at 7 to 9 with a layer, and grows with K.  Microseconds of a bf16 launch, few rows and tiles:
//   input gradient: 288 -> 96, 11 776 rows (26 496) 9.3 and 7.5; 192 -> 192, 7296 (21 888) 9.4 and 6.3; 48 -> 48, 38 528 (14 448) 10.3 and 7.2;
//   layers of whole steps of 64 channels: 192 -> 192, 7296 rows (21 888) 7.8 and 6.7; 384 -> 384, 2816 (33 792) 9.5 and 8.3; with GELU
//     later: 192 -> 768, 1920 rows (23 040) 8.5 and 9.3, 2688 (32 256) 10.0 and 9.9;
//   up to 96 channels: 48 -> 48 with a residual, 57 216 rows (21 456) 9.1 and 9.3, 76 160 (28 560) 11.9 and 9.5; with GELU 96 -> 384, 9984
//     (29 952) 11.0 and 13.0, 14 336 (43 008) 14.7 and 13.7; with fp32
//     results 96 -> 96, 39 936 (29 952) 10.7 and 11.5, 48 768 (36 576) 13.1 and 12.4;
//   others, whose last step is ragged in the tiles: 144 -> 144, 19 328 rows (43 488) 9.2 and 9.8; 240 -> 240, 5120 (28 800) 5.5 and 7.7;
//     480 -> 480, 2560 (48 000) 8.0 and 9.7; and fewer than 96 columns, which a tile does not use: 192 -> 48, 18 048 (27 072) 6.6 and 6.9.
// fp32 results of 16-bit rows show how they were summed (16-bit results differ by a rounding and have the same error, 2.1e-4 fp16 and
// 1.7e-3 bf16): with tiles only where their error against float64 is no larger, fp16 192 -> 192 5.3e-8 either way, but 288 -> 288
// 5.4e-8 and 5.9e-8, and behind 512 tiles, where a tile is summed in one part, 96 -> 96 4.8e-8 and 5.2e-8.
static int64_t few_line(int64_t N, int K, int P, int epi, bool down, bool wide) {
    if (wide && (K > 192 || (N + 127) / 128 * ((P + 95) / 96) > 512)) return FEW_MOST;
    if (down) return std::min<int64_t>(FEW_MOST, 12000 + 50 * K);
    if (P < 96 && K > 48) return FEW_MOST;
    if (K % 64 == 0) return std::min<int64_t>(FEW_MOST, (epi == EPI_GELU ? 22000 : 12000) + 50 * K);
    if (K <= 96) return epi == EPI_GELU ? 40000 : wide ? 35000 : 25000;
    return FEW_MOST;
}

template <typename T, typename TO, int EPI, bool DOWN>
static int launch_forward(const void* x, int64_t N, int K, const void* w, int P, const Epilogue& ep, float* ws, size_t ws_bytes, hipStream_t s) {
    const T* xp = static_cast<const T*>(x);
    const T* wp = static_cast<const T*>(w);
    if constexpr (Op<T>::PL == 1 && EPI == EPI_NONE && !DOWN)
        // not in place: its last tile reads rows again that another wavefront may have stored
        if (rows_once_takes(N, K, P) && ep.y != x) return rows_once<T>(xp, N, K, wp, static_cast<const T*>(ep.bias), P, static_cast<T*>(ep.y), s);
    const int64_t few_blocks = (N + 31) / 32 * ((P + 31) / 32);
    Cut cut = cut_of(Op<T>::PL == 3 ? SSWIN_F32 : SSWIN_F16, N, K, P, few_line(N, K, P, EPI, DOWN, sizeof(T) < sizeof(TO)));
    if (cut.few && few_blocks < (1ll << 31)) {
        hipLaunchKernelGGL((dense_small_kernel<T, TO, EPI, DOWN>), dim3((unsigned)few_blocks), dim3(SMALL_WAVES * 64), 0, s, xp, N, K, wp, P,
                           (P + 31) / 32, ep);
        return launch_ok("dense, few rows");
    }
    if constexpr (Op<T>::PL == 3) {
        // In place only dense_rows_kernel, which has read a row's values and formed what came out NaN again before it stores the first column: the
        // kernels of pairs store 32 columns at a time, that of tall_linear.hip reads rows of the last tile twice.
        const bool apart = ep.y != x;
        // 96 channels: the kernels that keep Wop in LDS
        if (apart && K == 96 && P % 96 == 0) {
            int rc = 0;
            if (pairs_held<EPI, DOWN>(xp, N, wp, P, ep, s, rc)) return rc;
            return staged_layer_96(xp, N, wp, P, DOWN, ep, s);
        }
        // fp16 pairs, from the reductions on whose sums come out as exactly: error against float64 (2-norms) with 96 channels 7.8e-8 and
        // 1.0e-7 here, 144 1.1e-7 and 1.75e-7 (turned); 48 channels of three bf16 pieces 6.9e-8, of pairs 7.1e-8 and more
        // The launch for W costs up to 2 us where tiles and reduction are few (three pieces and pairs, us): 9563 rows 112 -> 192 11.0 and 12.4, 4187 rows 144 -> 576
        // 12.5 and 13.6, 32 700 rows 144 -> 48 turned 13.3 and 14.0, 16 300 rows 192 -> 192 15.0 and 15.4; from 288 reduction channels on pairs are ahead everywhere.
        if (apart && pairs_takes(K) && ws_bytes >= pairs_workspace_bytes(K, P)) return pairs_layer<EPI, DOWN>(xp, N, K, wp, P, ep, ws, s);
        // 64 columns a workgroup and four wavefronts a SIMD, or 96 and three (what the registers allow without spilling).  Bound by the waits between request,
        // splitting and products of two or three short steps, so that the fourth wavefront counts, and by columns that a tile does not use.  96 -> 64, us, 112 700
        // rows from memory: 48 -> 48 19.7 -> 14.1, turned 17.4 -> 13.5, 48 -> 144 34.5 -> 32.6, 80 -> 48 25.7 -> 18.1; from the last-level cache: 48 -> 96 12.8 and
        // 12.4, 48 -> 128 17.4 -> 12.5, 80 -> 240 37.4 -> 33.3; with a residual 48 -> 96 20.7 -> 17.3, 80 -> 288 52.3 and 50.2.  Where 96 cover P with fewer columns and
        // there is no second operand they stay ahead: 48 -> 288 30.3 and 31.2, turned 26.7 and 28.2.  In place a workgroup has to hold whole rows.
        const bool wide = P > 96 && (P + 63) / 64 * 64 > (P + 95) / 96 * 96 && !Second4<float, float, EPI>::USED;
        if (apart && K < 96 && !wide) return launch_rows<EPI, DOWN, 4, 1, 2, 4>(xp, N, K, wp, P, ep, s);
        return launch_rows<EPI, DOWN, 4, 1, 3, 3>(xp, N, K, wp, P, ep, s);
    } else {
        if (ws_bytes < (size_t)cut.ksplit * N * P * sizeof(float)) cut.ksplit = 1;
        const int64_t rows = (N + 127) / 128, tiles = rows * ((P + 95) / 96) * cut.ksplit;
        // long reductions into many columns: fewest bytes through LDS (8119 rows, 768 -> 3072: 57 us against 70 with the next two)
        if (K >= 384 && P % 192 == 0 && rows * (P / 192) >= 512) return launch_rows16<T, TO, EPI, DOWN, 64, 2, 2, 1, 2, 2, 2>(xp, N, K, wp, P, 1, ws, ep, s);
        // one workgroup a compute unit and a long reduction: three blocks on their way instead of one, since nothing else hides a block's
        // way from L2 (five blocks of LDS where this has four: 7888 rows 1536 -> 384 22.0 us and 20.8).  bf16, other rows and weights in each call, with one
        // block and with three: 1364 rows 768 -> 768 14.7 and 11.6, 4000 rows 15.4 and 12.5, 8000 rows 768 -> 384 15.5 and 12.7, 7888 rows 1536 -> 384 28.2 and
        // 21.8, 700 rows 1536 -> 1536 21.4 and 18.7, 3000 rows 1024 -> 512 18.0 and 13.8.  With more tiles than compute units it loses: 7000 rows
        // 784 -> 400 (275) 19.9 and 25.0, 1364 rows 768 -> 3072 (352) 21.6 and 27.2.
        if (tiles <= device_cus() && K >= 768) return launch_rows16<T, TO, EPI, DOWN, 64, 4, 1, 2, 1, 4, 2>(xp, N, K, wp, P, cut.ksplit, ws, ep, s);
        // up to two workgroups a compute unit: eight wavefronts each (8119 rows, 1536 -> 384: 22 us against 30), above that five
        // workgroups of four, whose loads and stores overlap (219 000 rows, 96 -> 288: 44 us against 80)
        if (tiles <= 512) return launch_rows16<T, TO, EPI, DOWN, 64, 4, 1, 2, 1, 2, 4>(xp, N, K, wp, P, cut.ksplit, ws, ep, s);
        return launch_rows16<T, TO, EPI, DOWN, 32, 4, 1, 1, 1, 2, 5>(xp, N, K, wp, P, 1, ws, ep, s);
    }
}

template <typename T, typename TO>
static int pick_forward(int epi, bool down, const void* x, int64_t N, int K, const void* w, int P, const Epilogue& ep, float* ws, size_t ws_bytes, hipStream_t s) {
    if (down) {
        if (epi == EPI_NONE) return launch_forward<T, TO, EPI_NONE, true>(x, N, K, w, P, ep, ws, ws_bytes, s);
        return launch_forward<T, TO, EPI_SCALE, true>(x, N, K, w, P, ep, ws, ws_bytes, s);
    }
    if (epi == EPI_NONE) return launch_forward<T, TO, EPI_NONE, false>(x, N, K, w, P, ep, ws, ws_bytes, s);
    if (epi == EPI_GELU) return launch_forward<T, TO, EPI_GELU, false>(x, N, K, w, P, ep, ws, ws_bytes, s);
    return launch_forward<T, TO, EPI_RESIDUAL, false>(x, N, K, w, P, ep, ws, ws_bytes, s);
}

// fp32 parameters of a block in the tokens' type, one launch for all of them (a launch each: about 4 us x 8)
struct CastParts {
    const float* src[SSWIN_CAST_PARTS];
    int64_t first[SSWIN_CAST_PARTS + 1];                                 // of each in the destination, in pieces of 8 values
};
template <typename T> __global__ __launch_bounds__(256) void cast_parts_kernel(CastParts p, int count, T* __restrict__ dst) {
    const int64_t piece = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (piece >= p.first[count]) return;
    int which = 0;
    while (piece >= p.first[which + 1]) ++which;
    const f32x4* src = reinterpret_cast<const f32x4*>(p.src[which] + (piece - p.first[which]) * 8);
    const f32x4 a = src[0], b = src[1];
    u32x4 out;
    out[0] = pack2<T>(a[0], a[1]), out[1] = pack2<T>(a[2], a[3]), out[2] = pack2<T>(b[0], b[1]), out[3] = pack2<T>(b[2], b[3]);
    reinterpret_cast<u32x4*>(dst)[piece] = out;
}

// tiles of dW and row chunks: about `per_cu` workgroups per compute unit
struct WgradPlan {
    int tiles_p, tiles_k, chunks;
    int64_t rows;
};
static WgradPlan wgrad_plan(int64_t N, int P, int K, int bk, int min_rows, int bm, int bn, int per_cu) {
    WgradPlan p;
    p.tiles_p = (P + bm - 1) / bm;
    p.tiles_k = (K + bn - 1) / bn;
    const int64_t want = std::max<int64_t>(1, (int64_t)per_cu * device_cus() / ((int64_t)p.tiles_p * p.tiles_k));
    int64_t rows = std::max<int64_t>((N + want - 1) / want, min_rows);
    rows = (rows + bk - 1) / bk * bk;
    p.rows = rows;
    p.chunks = (int)((N + rows - 1) / rows);
    return p;
}

// rows up to which one launch of 32 x 32 tiles beats row chunks and their sums (284 rows 384 -> 1152: 19 us in chunks)
constexpr int64_t WGRAD_SMALL_ROWS = 1024;
// Tiles of dW.  fp32: by the columns it has, since a tile wider than dW works on copies of its last columns.
//   from 97 columns of X on 128 x 192, and 96 x 192 where that takes no more tiles (35 569 rows 192 -> 576: 64 us, with 96 x 192 61
//   but sums a fifth longer and 8 % more rounding; 192 -> 768 73, 192 -> 192 30, 768 -> 192 78; 75 000 rows 144 -> 144: 48 us, in tiles
//   of 128 x 96 56); 64 x 192 where dY has at most 64 (112 700 rows 192 -> 48: 37 us; 112 -> 48 31, in tiles of 128 x 96 46);
//   192 x 64 and 64 x 64 up to 64 columns of X (112 700 rows 48 -> 144 and 48 -> 48: 36 and 19 us);
//   128 x 96 between (75 000 rows 80 -> 112: 27 us).
// Rows of a sum (one row group of one chunk) decide the rounding as well: the matrix instructions do not round to nearest, what
// they leave is of one sign and grows with the number of sums, everything else with their length.  Relative error against float64
// of 30 000 rows 48 -> 48: sums of 32 rows 2.5e-7, of 64 2.1e-7; of 112 700 rows 144 -> 144: of 587 rows 5.7e-7, of 448 5.1e-7.
//   A sum has at least 64 rows.  Below 6144 rows (three row groups: 3072) sums are few, and shorter ones fill the chip: 4097 rows
//   48 -> 48 9.2 us and 1.3e-7, in sums of 64 rows 10.5 and 1.4e-7; but 6000 rows 80 -> 80 14.4 and 1.7e-7, 16.4 and 1.5e-7.
//   Tiles of 128 x 96 take two workgroups a compute unit where one would make sums longer than 128 rows and than tiles of 96 x 96
//   with four had: 112 700 rows 80 -> 80 34 us and 3.5e-7, with two 41 and 3.4e-7; 225 700 rows 53 and 5.5e-7, 62 and 4.5e-7.
// 16 bit: 96 x 96 (219 000 rows 96 -> 288: 39 us; 192 x 192 tiles 58, 192 x 96 44); 192 x 192 where dW has at least 48 such tiles
//   and the rows are many, so that half the bytes pass from L2 (8119 rows 768 -> 2304: 69 us and 57, 768 -> 3072 80 and 61;
//   2000 rows 768 -> 2304 25 and 26; 9000 rows 384 -> 1536 30 either way).
struct WgradTile {
    int bm, bn, per_cu, parts;                                           // fp32: row groups of a workgroup
};
static WgradTile wgrad_tile(int dtype, int64_t N, int P, int K) {
    if (dtype != SSWIN_F32) {
        if (N >= 4096 && P % 192 == 0 && K % 192 == 0 && (int64_t)P * K >= 48 * 192 * 192) return {192, 192, 1, 1};
        return {96, 96, 3, 1};
    }
    const int tall = (P + 127) / 128, low = (P + 95) / 96;
    if (K > 96) return P <= 64 ? WgradTile{64, 192, 2, 1} : tall < low ? WgradTile{128, 192, 1, 2} : WgradTile{96, 192, 1, 2};
    if (K <= 64) return P <= 64 ? WgradTile{64, 64, 2, 2} : WgradTile{192, 64, 1, 2};
    return {128, 96, 4 * tall <= 3 * low || N * tall <= (int64_t)3 * 128 * device_cus() ? 1 : 2, 3};
}
static WgradPlan wgrad_plan(int dtype, int64_t N, int P, int K) {
    const WgradTile t = wgrad_tile(dtype, N, P, K);
    if (dtype != SSWIN_F32) return wgrad_plan(N, P, K, 32, 128, t.bm, t.bn, t.per_cu);
    return wgrad_plan(N, P, K, 16, N < (t.parts == 2 ? 6144 : 3072) ? 64 : 64 * t.parts, t.bm, t.bn, t.per_cu);
}

template <typename T, typename TO, typename F>
static int launch_wgrad_as(F* k, int threads, size_t lds, const WgradPlan& pl, const void* dy, const void* x, int64_t N, int P, int K, void* dw, void* db,
                           float* ws, hipStream_t s) {
    float* part_b = ws + (size_t)pl.chunks * P * K;
    hipLaunchKernelGGL(k, dim3((unsigned)(pl.tiles_p * pl.tiles_k * pl.chunks)), dim3(threads), lds, s, static_cast<const T*>(dy), static_cast<const T*>(x), N,
                       P, K, pl.tiles_p, pl.tiles_k, pl.rows, ws, db ? part_b : nullptr);
    if (int rc = launch_ok("dense weight gradient")) return rc;
    const int64_t PK = (int64_t)P * K;
    const bool narrow = pl.chunks >= 256 || (sizeof(T) == 4 && pl.chunks >= 150 && PK <= 16384);
    if (pl.chunks <= 16)
        hipLaunchKernelGGL((dense_wgrad_sum_kernel<TO, 64>), dim3((unsigned)((PK + P + 255) / 256)), dim3(256), 0, s, ws, part_b, pl.chunks, PK, P,
                           static_cast<TO*>(dw), static_cast<TO*>(db));
    else if (narrow)
        hipLaunchKernelGGL((dense_wgrad_sum_kernel<TO, 4>), dim3((unsigned)((PK + P + 15) / 16)), dim3(256), 0, s, ws, part_b, pl.chunks, PK, P,
                           static_cast<TO*>(dw), static_cast<TO*>(db));
    else
        hipLaunchKernelGGL((dense_wgrad_sum_kernel<TO, 16>), dim3((unsigned)((PK + P + 63) / 64)), dim3(256), 0, s, ws, part_b, pl.chunks, PK, P,
                           static_cast<TO*>(dw), static_cast<TO*>(db));
    return launch_ok("dense weight gradient, sums");
}

// fp32: row groups of two buffers of (column tiles) x 3 planes
template <auto* KERNEL, typename TO>
static int launch_wgrad_f32(int waves, const WgradTile& t, const WgradPlan& pl, const void* dy, const void* x, int64_t N, int P, int K, void* dw,
                            void* db, float* ws, hipStream_t s) {
    const size_t lds = 2 * (size_t)t.parts * ((t.bm + t.bn) / 32) * 3 * 1024;
    static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void*>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    SSWIN_HIP(configured);
    return launch_wgrad_as<float, TO>(KERNEL, waves * 64, lds, pl, dy, x, N, P, K, dw, db, ws, s);
}

template <typename T, typename TO>
static int launch_wgrad(const void* dy, const void* x, int64_t N, int P, int K, void* dw, void* db, float* ws, hipStream_t s) {
    if (N <= WGRAD_SMALL_ROWS) {
        const int tp = (P + 31) / 32, tk = (K + 31) / 32;
        hipLaunchKernelGGL((dense_wgrad_small_kernel<T, TO>), dim3((unsigned)(tp * tk)), dim3(SMALL_WAVES * 64), 0, s, static_cast<const T*>(dy),
                           static_cast<const T*>(x), N, P, K, tk, static_cast<TO*>(dw), static_cast<TO*>(db));
        return launch_ok("dense weight gradient, few rows");
    }
    if constexpr (Op<T>::PL == 3) {
        const WgradPlan pl = wgrad_plan(SSWIN_F32, N, P, K);
        const WgradTile t = wgrad_tile(SSWIN_F32, N, P, K);
        if (t.bm == 128 && t.bn == 192) return launch_wgrad_f32<dense_wgrad_kernel<2, 3, 2, 2, 2, 3>, TO>(12, t, pl, dy, x, N, P, K, dw, db, ws, s);
        if (t.bm == 96) return launch_wgrad_f32<dense_wgrad_kernel<3, 2, 2, 1, 3, 3>, TO>(12, t, pl, dy, x, N, P, K, dw, db, ws, s);
        if (t.bn == 192) return launch_wgrad_f32<dense_wgrad_kernel<2, 2, 1, 1, 3, 2>, TO>(4, t, pl, dy, x, N, P, K, dw, db, ws, s);
        if (t.bm == 192) return launch_wgrad_f32<dense_wgrad_kernel<6, 1, 2, 1, 2, 3>, TO>(12, t, pl, dy, x, N, P, K, dw, db, ws, s);
        if (t.bm == 64) return launch_wgrad_f32<dense_wgrad_kernel<2, 1, 2, 1, 2, 3>, TO>(4, t, pl, dy, x, N, P, K, dw, db, ws, s);
        return launch_wgrad_f32<dense_wgrad_kernel<4, 1, 3, 1, 3, 3>, TO>(12, t, pl, dy, x, N, P, K, dw, db, ws, s);
    } else {
        constexpr size_t lds = 3 * 2 * 32 * 192;                         // three stages of two tiles of 32 x 96
        const WgradPlan pl = wgrad_plan(SSWIN_F16, N, P, K);
        if (wgrad_tile(SSWIN_F16, N, P, K).bm == 192) {
            auto* k = dense16_wgrad_kernel<T, 3, 2, 2, 3, 2>;
            static const int configured = allow_lds(k, 2 * lds);
            if (configured) return configured;
            return launch_wgrad_as<T, TO>(k, 384, 2 * lds, pl, dy, x, N, P, K, dw, db, ws, s);
        }
        return launch_wgrad_as<T, TO>(dense16_wgrad_kernel<T, 3, 1, 1, 3, 3>, 192, lds, pl, dy, x, N, P, K, dw, db, ws, s);
    }
}

template <typename T, typename TO>
static int launch_backward_small(int epi, const void* dy, const void* x, const void* w, int64_t N, int P, int K, const Epilogue& ep, void* dw, void* db,
                                 hipStream_t s) {
    const int tiles_k = (K + 31) / 32, dx_tiles = (int)((N + 31) / 32) * tiles_k, dw_tiles = (P + 31) / 32 * tiles_k;
    const dim3 grid((unsigned)(dx_tiles + dw_tiles)), block(SMALL_WAVES * 64);
    if (epi == EPI_SCALE)
        hipLaunchKernelGGL((dense_backward_small_kernel<T, TO, EPI_SCALE>), grid, block, 0, s, static_cast<const T*>(dy), static_cast<const T*>(x),
                           static_cast<const T*>(w), N, P, K, dx_tiles, tiles_k, ep, static_cast<TO*>(dw), static_cast<TO*>(db));
    else
        hipLaunchKernelGGL((dense_backward_small_kernel<T, TO, EPI_NONE>), grid, block, 0, s, static_cast<const T*>(dy), static_cast<const T*>(x),
                           static_cast<const T*>(w), N, P, K, dx_tiles, tiles_k, ep, static_cast<TO*>(dw), static_cast<TO*>(db));
    return launch_ok("dense backward, few rows");
}

}  // namespace dense
}  // namespace sswin

using namespace sswin;
using namespace sswin::dense;

extern "C" {

int sswin_dense_supported(int dtype, int P, int K) {
    return (dtype == SSWIN_F32 || dtype == SSWIN_F16 || dtype == SSWIN_BF16) && P > 0 && K > 0 && P % 16 == 0 && K % 16 == 0;
}

size_t sswin_dense_forward_workspace_bytes(int dtype, int64_t N, int K, int P) {
    if (N <= 0 || !sswin_dense_supported(dtype, P, K)) return 0;
    const Cut c = cut_of(dtype, N, K, P);
    if (dtype == SSWIN_F32) return c.few || !pairs_takes(K) || (K == 96 && P % 96 == 0) ? 0 : pairs_workspace_bytes(K, P);
    return c.ksplit > 1 ? (size_t)c.ksplit * N * P * sizeof(float) : 0;
}

int sswin_dense_forward(int dtype, int out_dtype, int transposed, int epilogue, const void* x, int64_t N, int K, const void* w, const void* bias,
                        int P, const void* extra, void* y, void* slope, void* ws, size_t ws_bytes, void* stream) {
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
    SSWIN_CHECK(((uintptr_t)ws) % 16 == 0, "dense_forward: the workspace must be 16-byte aligned");
    if (!ws) ws_bytes = 0;                                               // whatever size goes with a null pointer
    float* f = static_cast<float*>(ws);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool down = transposed != 0;
#define DENSE_RUN(T, TO) return pick_forward<T, TO>(epilogue, down, x, N, K, w, P, ep, f, ws_bytes, s)
    if (dtype == SSWIN_F32 && out_dtype == SSWIN_F32) DENSE_RUN(float, float);
    if (dtype == SSWIN_F16 && out_dtype == SSWIN_F16) DENSE_RUN(__half, __half);
    if (dtype == SSWIN_BF16 && out_dtype == SSWIN_BF16) DENSE_RUN(__hip_bfloat16, __hip_bfloat16);
    if (epilogue == EPI_RESIDUAL) {                                      // mixed precision: the residual stream stays fp32
        if (dtype == SSWIN_F16 && out_dtype == SSWIN_F32) return launch_forward<__half, float, EPI_RESIDUAL, false>(x, N, K, w, P, ep, f, ws_bytes, s);
        if (dtype == SSWIN_BF16 && out_dtype == SSWIN_F32)
            return launch_forward<__hip_bfloat16, float, EPI_RESIDUAL, false>(x, N, K, w, P, ep, f, ws_bytes, s);
    }
#undef DENSE_RUN
    return fail("dense_forward: operands of type %d with a result of type %d are not supported", dtype, out_dtype);
}

int sswin_cast_parts(int dtype, const void* const* src, const int64_t* sizes, int count, void* dst, void* stream) {
    SSWIN_CHECK(count >= 1 && count <= SSWIN_CAST_PARTS && src && sizes && dst, "cast_parts: 1 to %d parts", SSWIN_CAST_PARTS);
    SSWIN_CHECK(dtype == SSWIN_F16 || dtype == SSWIN_BF16, "cast_parts: type %d", dtype);
    CastParts p;
    p.first[0] = 0;
    for (int i = 0; i < count; ++i) {
        SSWIN_CHECK(src[i] && sizes[i] >= 0 && sizes[i] % 8 == 0 && (uintptr_t)src[i] % 16 == 0, "cast_parts: parts are multiples of 8 values, 16-byte aligned");
        p.src[i] = static_cast<const float*>(src[i]);
        p.first[i + 1] = p.first[i] + sizes[i] / 8;
    }
    SSWIN_CHECK((uintptr_t)dst % 16 == 0, "cast_parts: pointers must be 16-byte aligned");
    const int64_t blocks = (p.first[count] + 255) / 256;
    SSWIN_CHECK(blocks < (1ll << 31), "cast_parts: too many values");
    if (blocks == 0) return 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == SSWIN_F16) hipLaunchKernelGGL((cast_parts_kernel<__half>), dim3((unsigned)blocks), dim3(256), 0, s, p, count, static_cast<__half*>(dst));
    else hipLaunchKernelGGL((cast_parts_kernel<__hip_bfloat16>), dim3((unsigned)blocks), dim3(256), 0, s, p, count, static_cast<__hip_bfloat16*>(dst));
    return launch_ok("cast_parts");
}

int sswin_dense_backward_small_supported(int dtype, int64_t N, int P, int K) {
    // where both gradients would take their few-rows kernels; 16 bit: also where dX alone would not, since it saves a launch
    if (N <= 0 || N > WGRAD_SMALL_ROWS || !sswin_dense_supported(dtype, P, K)) return 0;
    return dtype == SSWIN_F32 ? cut_of(dtype, N, P, K).few : (N + 127) / 128 * ((K + 95) / 96) * P <= 50000;
}

int sswin_dense_backward_small(int dtype, int out_dtype, int epilogue, const void* dy, const void* x, const void* w, int64_t N, int P, int K,
                               const void* extra, void* dx, void* dw, void* db, void* stream) {
    SSWIN_CHECK(sswin_dense_backward_small_supported(dtype, N, P, K), "dense_backward_small: %lld rows, %d -> %d channels of type %d are not supported",
                (long long)N, K, P, dtype);
    SSWIN_CHECK(epilogue == EPI_NONE || (epilogue == EPI_SCALE && extra), "dense_backward_small: epilogue %d", epilogue);
    SSWIN_CHECK(dy && x && w && dx && dw, "dense_backward_small: null pointer");
    SSWIN_CHECK(((uintptr_t)dy | (uintptr_t)x | (uintptr_t)w | (uintptr_t)extra | (uintptr_t)dx | (uintptr_t)dw | (uintptr_t)db) % 16 == 0,
                "dense_backward_small: pointers must be 16-byte aligned");
    const Epilogue ep = {nullptr, extra, dx, nullptr};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == SSWIN_F32 && out_dtype == SSWIN_F32) return launch_backward_small<float, float>(epilogue, dy, x, w, N, P, K, ep, dw, db, s);
    if (dtype == SSWIN_F16 && out_dtype == SSWIN_F16) return launch_backward_small<__half, __half>(epilogue, dy, x, w, N, P, K, ep, dw, db, s);
    if (dtype == SSWIN_F16 && out_dtype == SSWIN_F32) return launch_backward_small<__half, float>(epilogue, dy, x, w, N, P, K, ep, dw, db, s);
    if (dtype == SSWIN_BF16 && out_dtype == SSWIN_BF16)
        return launch_backward_small<__hip_bfloat16, __hip_bfloat16>(epilogue, dy, x, w, N, P, K, ep, dw, db, s);
    if (dtype == SSWIN_BF16 && out_dtype == SSWIN_F32) return launch_backward_small<__hip_bfloat16, float>(epilogue, dy, x, w, N, P, K, ep, dw, db, s);
    return fail("dense_backward_small: operands of type %d with gradients of type %d are not supported", dtype, out_dtype);
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
