// fp32 dense layers of at least 96 reduction channels on the fp16 matrix cores, every operand as two fp16 pieces (Pairs of
// dense_operand.hpp): y [N, P] = last step of x [N, K] Wop, as dense_rows_kernel of dense.hip, which takes shorter reductions, and calls
// without a workspace.
//
// A launch of its own splits W, once for all rows: its pieces lie in the workspace in operand order, scaled by a power of two per
// column, and pass from there to LDS without registers.  A wavefront owns 32 rows and 96 columns.  Its rows pass to its own part of
// LDS as they are, a step of 32 columns at a time (whole lines, the next step requested as soon as this one is in registers: no
// barrier, no second buffer), and are split in operand order, where a lane holds one row: the row's scale is one number a lane.  It
// follows the largest value seen so far: where a step's values would leave fp16's range the row's scale drops and what has been summed
// drops with it.  Products are formed transposed (rows of the result: columns of y), so that a row's sums lie in that row's lanes as well.
//
// Microseconds with the launch for W, and as three bf16 pieces before: 35 569 rows 192 -> 576 45 and 62, 576 -> 192 turned 42 and 64, 768 -> 192 with a
// residual 54 and 79, 192 -> 768 turned with a factor 62 and 87; 112 700 rows 288 -> 96 turned 36 and 50; 9000 rows 768 -> 2304 126 and 192, 1536 -> 384
// turned 60 and 91.  Error against float64 (2-norms): K = 192 8.8e-8 and 1.4e-7, 576 1.7e-7 and 3.6e-7, 1536 2.6e-7 and 6.0e-7.
// 768 -> 2304: the matrix cores are busy for 40 % of the launch; without the loads it takes 80 % of its time, without the products 72 %, with neither
// and no splitting 41 %: three wavefronts a SIMD, each a chain of reads, splitting and products between two barriers.  Not ahead: 64 rows a
// wavefront (45 -> 52, 126 -> 127), 256 rows or 192 columns a workgroup (45 -> 48 and 47), two to four steps in flight (45 -> 53, 126 -> 134), the
// splitting one step ahead between the products at two wavefronts a SIMD (45 -> 57, 126 -> 146), rows kept in registers for all columns (45 -> 49 to 55).
#include <stdint.h>

#include <algorithm>

#include "dense_epilogue.hpp"
#include "dense_operand.hpp"
#include "mfma_block.hpp"
#include "sswin_common.hpp"

namespace sswin {
namespace dense {

__host__ __device__ static constexpr int pairs_ksteps(int K) { return (K + 31) / 32 * 2; }

// Pieces of W in operand order, [column tile of 32][step of 16 channels][piece][lane], and the exponents of the columns' scales; columns
// past the last repeat it, the half of the last step of 32 that K ends before is zero.  What such a launch takes is latency, so the columns go to
// as many compute units as they can: W [P, K] a wavefront a column, 512 of its values at a time, the first 1536 kept in registers (192 -> 576
// 5.0 us in workgroups of 32 columns, 768 -> 2304 9.7); W [K, P] (DOWN) a workgroup for 32 columns.
template <bool DOWN>
__global__ __launch_bounds__(DOWN ? 1024 : 256) void pairs_weights_kernel(const float* __restrict__ w, int K, int P, u32x4* __restrict__ planes,
                                                                         int* __restrict__ exps) {
    const int ksteps = pairs_ksteps(K);
    auto at = [&](int col, int ks, int half) { return planes + ((int64_t)(col >> 5) * ksteps + ks) * 128 + half * 32 + (col & 31); };
    if constexpr (DOWN) {
        const int e = pairs_of_columns<true, 16, false>(w, K, P, blockIdx.x, [&](int col, int ks, int half, const u32x4 (&p)[2]) {
            u32x4* dst = at(col, ks, half);
            dst[0] = p[0];
            dst[64] = p[1];
        });
        if (threadIdx.x < 128 && ksteps > K / 16) planes[((int64_t)blockIdx.x * ksteps + K / 16) * 128 + threadIdx.x] = u32x4{0, 0, 0, 0};
        if (threadIdx.x < 32) exps[blockIdx.x * 32 + threadIdx.x] = e;
    } else {
        constexpr int KEPT = 3;
        const int col = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
        const float* const row = w + (int64_t)min(col, P - 1) * K + lane * 8;
        const int own = (K - lane * 8 + 511) / 512;                      // rounds of 512 in which this lane has eight values
        auto load = [&](int i, float (&v)[8]) {
            const f32x4 a = *reinterpret_cast<const f32x4*>(row + i * 512), b = *reinterpret_cast<const f32x4*>(row + i * 512 + 4);
#pragma unroll
            for (int c = 0; c < 8; ++c) v[c] = c < 4 ? a[c] : b[c - 4];
        };
        float kept[KEPT][8], m = 0.f;
#pragma unroll
        for (int i = 0; i < KEPT; ++i)
            if (i < own) load(i, kept[i]);
#pragma unroll
        for (int i = 0; i < KEPT; ++i)
            if (i < own) m = fmaxf(m, largest(kept[i]));
        for (int i = KEPT; i < own; ++i) {
            float v[8];
            load(i, v);
            m = fmaxf(m, largest(v));
        }
        m = largest_of_halves(row16_max(m));
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        const int e = pairs_scale(exponent_above(m));
        const float scale = power_of_two(e);
        auto put = [&](int i, const float (&v)[8]) {
            u32x4 p[2];
            split_pairs(v, scale, p);
            u32x4* dst = at(col, i * 32 + lane / 2, lane & 1);
            dst[0] = p[0];
            dst[64] = p[1];
        };
#pragma unroll
        for (int i = 0; i < KEPT; ++i)
            if (i < own) put(i, kept[i]);
        for (int i = KEPT; i < own; ++i) {
            float v[8];
            load(i, v);
            put(i, v);
        }
        if (ksteps > K / 16 && lane < 4) at(col, K / 16, lane >> 1)[(lane & 1) * 64] = u32x4{0, 0, 0, 0};
        if (lane == 0) exps[col] = e;
    }
}

// The results of a wavefront's tile of 32 x 32 whose bits are set in `mask` (of lane l, register r: row l % 32, column 8 (r / 4) + 4 (l / 32) + r % 4)
// from product(row, column); true: they are many, and marked with NaN instead
template <typename F> __device__ __forceinline__ bool small_again(u32x4* tile, uint32_t mask, F product) {
    const int lane = threadIdx.x & 63;
    if (!__any(mask)) return false;
    auto at = [&](int l, int r) { return reinterpret_cast<float*>(tile + (l & 31) * 8 + ((r / 4 * 2 + (l >> 5)) ^ (l & 7))) + r % 4; };
    const bool many = many_small(mask);
    if (many) {
        for (; mask; mask &= mask - 1) *at(lane, __builtin_ctz(mask)) = NAN;
    } else {
        for_each_small(mask, [&](int owner, int r) {
            const float v = product(owner & 31, r / 4 * 8 + (owner >> 5) * 4 + r % 4);
            if (lane == owner) *at(lane, r) = v;
        });
    }
    __builtin_amdgcn_wave_barrier();
    return many;
}

template <int EPI, bool DOWN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void pairs_rows_kernel(
    const float* __restrict__ x, int64_t N, int K, const u32x4* __restrict__ planes, const int* __restrict__ exps, const float* __restrict__ w, int P,
    int groups, Epilogue ep) {
    constexpr int NT = 3, BN = NT * 32, WAVES = 4, BM = WAVES * 32, STEP_W = NT * 4 * 64;   // 16-byte pieces of W a step of 32 channels
    __shared__ __attribute__((aligned(16))) u32x4 lds[2 * STEP_W + WAVES * 256];                         // 40 KB
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    int cg;
    int64_t rb;
    block_of(groups, cg, rb);
    const int64_t row0 = rb * BM + wave * 32;
    const int col0 = cg * BN, steps = (K + 31) / 32, ksteps = pairs_ksteps(K);
    u32x4* const tile = lds + 2 * STEP_W + wave * 256;                   // [32 rows][8 pieces], the pieces of a row exchanged by its number

    const int piece = (lane & 7) ^ (lane >> 3);                          // of x, that this lane brings
    uint32_t ox[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t row = row0 + i * 8 + (lane >> 3);
        ox[i] = (uint32_t)((int)((row < N ? row : N - 1) - rb * BM) * K + piece * 4);   // rows past the end repeat the last one
    }
    const float* const xb = x + rb * BM * K;
    const u32x4* const wb = planes + (int64_t)cg * NT * ksteps * 128 + lane;
    auto request_x = [&](int step) {
        const int back = step * 32 + 16 == K && piece >= 4 ? 16 : 0;     // only 16 columns left: the upper half repeats them, and meets zeros
#pragma unroll
        for (int i = 0; i < 4; ++i) copy_to_lds(xb + step * 32 + (ox[i] - back), lds_address(tile + i * 64));
    };
    auto request_w = [&](int step) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int p = i * WAVES + wave;                              // [column tile][16 channels][piece]
            copy_to_lds(wb + ((int64_t)(p >> 2) * ksteps + step * 2) * 128 + (p & 3) * 64, lds_address(lds + (step & 1) * STEP_W + p * 64));
        }
    };
    request_w(0);
    request_x(0);

    f32x16 acc[NT], low[NT];                                             // (h,h); (l,h) and (h,l)
    int e = PAIRS_ZEROS_SO_FAR;                                          // exponent of the row's scale
    float scale = 0.f;
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = low[j] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int step = 0; step < steps; ++step) {
        wait_copies<0>();
        block_barrier();                                                 // this step's pieces are there, those of the last one have been read
        if (step + 1 < steps) request_w(step + 1);
        float v[2][8];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const f32x4 t = __builtin_bit_cast(f32x4, tile[l32 * 8 + ((h * 4 + half * 2 + q) ^ (l32 & 7))]);
#pragma unroll
                for (int c = 0; c < 4; ++c) v[h][q * 4 + c] = t[c];
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");               // read, so that the next step may come in its place
        if (step + 1 < steps) request_x(step + 1);
        const int above = exponent_above(largest_of_halves(fmaxf(largest(v[0]), largest(v[1]))));
        if (__any(above + e > 15)) {                                     // first step, or 4 times larger than what had been seen
            const int now = pairs_scale_after(above, e);
            const float factor = power_of_two(now - e);
            e = now, scale = power_of_two(min(now, PAIRS_MOST_SCALE));     // (rows of zeros so far too)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[j][r] *= factor, low[j][r] *= factor;
        }
        const u32x4* const pieces = lds + (step & 1) * STEP_W + lane;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 a[NT][2], b[2];
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int q = 0; q < 2; ++q) a[j][q] = pieces[((j * 2 + h) * 2 + q) * 64];
            split_pairs(v[h], scale, b);
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                low[j] = Pairs::mfma(a[j][1], b[0], low[j]);
                acc[j] = Pairs::mfma(a[j][0], b[0], acc[j]);
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) low[j] = Pairs::mfma(a[j][0], b[1], low[j]);
        }
    }
    // 32 rows x 32 columns at a time through the wavefront's part of LDS, so that memory is touched in runs of 128 bytes
    const int mem_row = lane >> 3, mem_col = ((lane & 7) ^ (lane >> 3)) * 4;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int col = col0 + j * 32 + mem_col;
            const int64_t r0 = row0 + mem_row;
            Second4<float, float, EPI> second[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (r0 + q * 8 < N && col < P) second[q].load(ep, r0 + q * 8, col, P);
            float least = INFINITY;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int4 ew = *reinterpret_cast<const int4*>(exps + col0 + j * 32 + q * 8 + half * 4);
                const int c[4] = {ew.x, ew.y, ew.z, ew.w};
                f32x4 t;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float s = fmaf(low[j][q * 4 + u], Pairs::LOW, acc[j][q * 4 + u]);
                    least = least_size(least, s);
                    t[u] = __builtin_amdgcn_ldexpf(s, -(e + c[u]));
                }
                tile[l32 * 8 + ((q * 2 + half) ^ (l32 & 7))] = __builtin_bit_cast(u32x4, t);
            }
            __builtin_amdgcn_wave_barrier();
            f32x4 y[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) y[q] = __builtin_bit_cast(f32x4, tile[q * 64 + lane]);
            if (__any(nan_or_small(least, e))) {
                uint32_t mask = 0;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int at = col0 + j * 32 + r / 4 * 8 + half * 4 + r % 4;
                    if (fabsf(fmaf(low[j][r], Pairs::LOW, acc[j][r])) < PAIRS_SMALL && at < P && exps[at] <= PAIRS_MOST_SCALE) mask |= 1u << r;
                }
                if (e > PAIRS_MOST_SCALE || row0 + l32 >= N) mask = 0;
                const bool many = small_again(tile, mask, [&](int r32, int c32) {
                    const int at = col0 + j * 32 + c32;
                    return wave_product(x + (row0 + r32) * K, w + (DOWN ? at : (int64_t)at * K), DOWN ? P : 1, K);
                });
                if (__any(least != least) || many) {
#pragma unroll 1
                    for (int q = 0; q < 4; ++q) {
                        f32x4 t = __builtin_bit_cast(f32x4, tile[q * 64 + lane]);
                        if (r0 + q * 8 < N && col < P && nan_among(t))
                            t = plain_products(x + (r0 + q * 8) * K, 1, w + (DOWN ? col : (int64_t)col * K), DOWN ? P : 1, DOWN ? 1 : K, K);
                        tile[q * 64 + lane] = __builtin_bit_cast(u32x4, t);
                    }
                    __builtin_amdgcn_wave_barrier();
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) y[q] = __builtin_bit_cast(f32x4, tile[q * 64 + lane]);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (r0 + q * 8 < N && col < P) finish4<float, float, EPI>(ep, r0 + q * 8, col, P, y[q], second[q]);
        }
}

// ------------------------------------------------------------------------------------------
// 96 reduction channels: a workgroup of 8 wavefronts a compute unit splits its 32 CT columns of W itself, keeps their pieces in LDS and walks over the
// rows, 32 a wavefront, the next 32 in flight.  A row's 96 values fit a lane as pieces (48 registers), so that its scale is that of its
// largest value and it is split once for all of the columns.  Bound by the traffic, and by what a launch takes until its pieces are there (5 us).
// The loops over the columns are unrolled: with a count the compiler does not know it waits for all stores where the next rows are used (CT = 9 in a
// loop 42 us where three workgroups of 96 columns take 39; unrolled, 36 registers are spilled and 50).
// Three bf16 pieces before, microseconds: 112 700 rows 96 -> 288 44.2 and 41.0, 96 -> 96 21.1 and 19.3 (turned 21.1 and 20.1), 225 700 rows 96 -> 288 87.3 and
// 87.5; with other rows and weights in each call 50 000 rows 96 -> 288 33.8 and 28.5, 96 -> 96 15.2 and 14.5 (turned 15.2 and 15.7), 20 000 rows 14.2 and 13.8,
// 10.6 and 8.3 (turned 10.8 and 8.9).  Inside an attention module, where rows and weights come from memory, the launches of 20 000 rows take 17.0 and 9.3 (before 26.0 together).
// Error against float64 (2-norms) 1.13e-7 and 0.81e-7, turned 1.50e-7 and 1.04e-7.  Not ahead: W's columns dealt to all wavefronts 16 channels at a time, their
// maxima through LDS (6400 rows 96 -> 288 8.2 -> 8.5, 20 000 13.6 -> 14.5, 51 200 28.7 -> 29.7).
// ------------------------------------------------------------------------------------------
constexpr int HELD_K = 96, HELD_KS = HELD_K / 16, HELD_WAVES = 8;
template <int EPI, bool DOWN, int CT>
__global__ __launch_bounds__(HELD_WAVES * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void pairs_held_kernel(
    const float* __restrict__ x, int64_t N, const float* __restrict__ w, int P, int groups, int64_t row_tiles, Epilogue ep) {
    constexpr int K = HELD_K, KS = HELD_KS;
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];          // pieces [column tile][16 channels][piece][lane], a tile a wavefront
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    int cg;
    int64_t slot;
    block_of(groups, cg, slot);
    const int col0 = cg * CT * 32;
    u32x4* const tile = lds + CT * KS * 128 + wave * 256;                // [32 rows][8 pieces], the pieces of a row exchanged by its number
    int* const exps = reinterpret_cast<int*>(lds + CT * KS * 128 + HELD_WAVES * 256);
    float* const bias = reinterpret_cast<float*>(exps + CT * 32);
    const int64_t first = slot * HELD_WAVES + wave, stride = (int64_t)(gridDim.x / groups) * HELD_WAVES;

    const int mem_row = lane >> 3, mem_piece = (lane & 7) ^ mem_row;     // of 8 rows x 32 columns, that this lane moves
    f32x4 next[3][4];
    auto fetch = [&](int64_t t) {                                        // rows past the end repeat the last one
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int64_t row = t * 32 + i * 8 + mem_row;
            const float* const from = x + (row < N ? row : N - 1) * K + mem_piece * 4;
#pragma unroll
            for (int c = 0; c < 3; ++c) next[c][i] = *reinterpret_cast<const f32x4*>(from + c * 32);
        }
    };
    if (first < row_tiles) fetch(first);
    if (const int c = wave; c < CT) {
        const int col = col0 + c * 32 + l32;
        float v[KS][8], m = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = ks * 16 + half * 8;
            if constexpr (DOWN) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[ks][e] = w[(int64_t)(k + e) * P + col];
            } else {
                const f32x4* const src = reinterpret_cast<const f32x4*>(w + (int64_t)col * K + k);
                const f32x4 a = src[0], b = src[1];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[ks][e] = e < 4 ? a[e] : b[e - 4];
            }
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) m = fmaxf(m, largest(v[ks]));
        const int e = pairs_scale(exponent_above(largest_of_halves(m)));
        const float scale = power_of_two(e);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            u32x4 p[2];
            split_pairs(v[ks], scale, p);
            lds[((c * KS + ks) * 2 + 0) * 64 + lane] = p[0];
            lds[((c * KS + ks) * 2 + 1) * 64 + lane] = p[1];
        }
        if (half == 0) {
            exps[c * 32 + l32] = e;
            bias[c * 32 + l32] = ep.bias ? static_cast<const float*>(ep.bias)[col] : 0.f;
        }
    }
    block_barrier();
    const Epilogue after = {nullptr, ep.extra, ep.y, ep.slope};          // the bias is added before
    for (int64_t t = first; t < row_tiles; t += stride) {
        float v[KS][8], m = 0.f;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < 4; ++i) tile[(i * 8 + mem_row) * 8 + (lane & 7)] = __builtin_bit_cast(u32x4, next[c][i]);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const f32x4 p = __builtin_bit_cast(f32x4, tile[l32 * 8 + ((h * 4 + half * 2 + q) ^ (l32 & 7))]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[c * 2 + h][q * 4 + e] = p[e];
                }
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) m = fmaxf(m, largest(v[ks]));
        const int e = pairs_scale(exponent_above(largest_of_halves(m)));
        const float scale = power_of_two(e);
        u32x4 b[KS][2];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) split_pairs(v[ks], scale, b[ks]);
        if (t + stride < row_tiles) fetch(t + stride);
        const int64_t r0 = t * 32 + mem_row;
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int col = col0 + c * 32 + mem_piece * 4;
            Second4<float, float, EPI> second[4];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (r0 + q * 8 < N) second[q].load(ep, r0 + q * 8, col, P);
            const u32x4* const pieces = lds + c * KS * 128 + lane;
            f32x16 acc = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}, low = acc;
            u32x4 a[2][2];
#pragma unroll
            for (int q = 0; q < 2; ++q) a[0][q] = pieces[q * 64];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                if (ks + 1 < KS)
#pragma unroll
                    for (int q = 0; q < 2; ++q) a[(ks + 1) & 1][q] = pieces[((ks + 1) * 2 + q) * 64];
                low = Pairs::mfma(a[ks & 1][1], b[ks][0], low);
                acc = Pairs::mfma(a[ks & 1][0], b[ks][0], acc);
                low = Pairs::mfma(a[ks & 1][0], b[ks][1], low);
            }
            float least = INFINITY;
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int at = c * 32 + q * 8 + half * 4;
                const int4 ew = *reinterpret_cast<const int4*>(exps + at);
                const f32x4 add = *reinterpret_cast<const f32x4*>(bias + at);
                const int ec[4] = {ew.x, ew.y, ew.z, ew.w};
                f32x4 s;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float p = fmaf(low[q * 4 + u], Pairs::LOW, acc[q * 4 + u]);
                    least = least_size(least, p);
                    s[u] = __builtin_amdgcn_ldexpf(p, -(e + ec[u])) + add[u];
                }
                tile[l32 * 8 + ((q * 2 + half) ^ (l32 & 7))] = __builtin_bit_cast(u32x4, s);
            }
            __builtin_amdgcn_wave_barrier();
            if (__any(nan_or_small(least, e))) {
                uint32_t mask = 0;
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (fabsf(fmaf(low[r], Pairs::LOW, acc[r])) < PAIRS_SMALL && exps[c * 32 + r / 4 * 8 + half * 4 + r % 4] <= PAIRS_MOST_SCALE) mask |= 1u << r;
                if (e > PAIRS_MOST_SCALE || t * 32 + l32 >= N) mask = 0;
                const bool many = small_again(tile, mask, [&](int r32, int c32) {
                    const int at = col0 + c * 32 + c32;
                    return wave_product(x + (t * 32 + r32) * K, w + (DOWN ? at : (int64_t)at * K), DOWN ? P : 1, K) + bias[c * 32 + c32];
                });
                if (__any(least != least) || many) {
#pragma unroll 1
                    for (int q = 0; q < 4; ++q) {
                        f32x4 s = __builtin_bit_cast(f32x4, tile[q * 64 + lane]);
                        if (r0 + q * 8 < N && nan_among(s))
                            s = plain_products(x + (r0 + q * 8) * K, 1, w + (DOWN ? col : (int64_t)col * K), DOWN ? P : 1, DOWN ? 1 : K, K) +
                                *reinterpret_cast<const f32x4*>(bias + (col - col0));
                        tile[q * 64 + lane] = __builtin_bit_cast(u32x4, s);
                    }
                    __builtin_amdgcn_wave_barrier();
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (r0 + q * 8 < N)
                    finish4<float, float, EPI>(after, r0 + q * 8, col, P, __builtin_bit_cast(f32x4, tile[q * 64 + lane]), second[q]);
        }
    }
}

static int pairs_tiles(int P) { return (P + 95) / 96 * 3; }
size_t pairs_workspace_bytes(int K, int P) { return (size_t)pairs_tiles(P) * (pairs_ksteps(K) * 2048 + 128); }

template <int EPI, bool DOWN> int pairs_layer(const float* x, int64_t N, int K, const float* w, int P, const Epilogue& ep, void* ws, hipStream_t s) {
    const int groups = (P + 95) / 96;
    const int64_t blocks = (N + 127) / 128 * groups;
    SSWIN_CHECK(blocks < (1ll << 31), "dense: too many rows");
    u32x4* planes = static_cast<u32x4*>(ws);
    int* exps = reinterpret_cast<int*>(planes + (size_t)pairs_tiles(P) * pairs_ksteps(K) * 128);
    const dim3 grid((unsigned)pairs_tiles(P) * (DOWN ? 1 : 8)), block(DOWN ? 1024 : 256);
    hipLaunchKernelGGL((pairs_weights_kernel<DOWN>), grid, block, 0, s, w, K, P, planes, exps);
    if (int rc = launch_ok("dense, pieces of the weights")) return rc;
    hipLaunchKernelGGL((pairs_rows_kernel<EPI, DOWN>), dim3((unsigned)blocks), dim3(256), 0, s, x, N, K, planes, exps, w, P, groups, ep);
    return launch_ok("dense, pairs");
}
template <int EPI, bool DOWN, int CT> static int launch_held(const float* x, int64_t N, const float* w, int P, const Epilogue& ep, hipStream_t s) {
    auto* k = pairs_held_kernel<EPI, DOWN, CT>;
    constexpr int LDS = CT * (HELD_KS * 2048 + 256) + HELD_WAVES * 4096;
    static const hipError_t configured = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    SSWIN_HIP(configured);
    const int groups = P / 32 / CT;
    const int64_t row_tiles = (N + 31) / 32, slots = std::min<int64_t>((row_tiles + HELD_WAVES - 1) / HELD_WAVES, std::max(1, device_cus() / groups));
    hipLaunchKernelGGL(k, dim3((unsigned)(slots * groups)), dim3(HELD_WAVES * 64), LDS, s, x, N, w, P, groups, row_tiles, ep);
    return launch_ok("dense, pairs of 96 channels");
}
// False where tall_linear.hip is ahead: its kernel requests a second operand when the products are done, here it stands behind the next
// rows, and in front of them there are no registers for it (112 700 rows 96 -> 96 with a residual: 21.2 us there, 23.3 here, in front 32).
template <int EPI, bool DOWN> bool pairs_held(const float* x, int64_t N, const float* w, int P, const Epilogue& ep, hipStream_t s, int& rc) {
    const int64_t workgroups = (N + HELD_WAVES * 32 - 1) / (HELD_WAVES * 32) * (P / 96);   // of 96 columns
    // few of them: 32 columns.  With 32 and with 96, other rows and weights in each call: 84 workgroups (7000 rows 96 -> 288) 8.3 and 11.1 us, 120 11.2 and 11.6,
    // 141 (36 000 rows 96 -> 96) 12.0 and 12.7, 160 (10 000 rows 96 -> 384) 11.8 and 12.0; 172 (22 000 rows 96 -> 192) 14.3 and 12.4, 196 15.3 and 13.1, 237
    // 16.0 and 13.8
    const bool few = workgroups * 8 <= device_cus() * 5;
    if (Second4<float, float, EPI>::USED && !few) return false;
    if constexpr (Second4<float, float, EPI>::USED) rc = launch_held<EPI, DOWN, 1>(x, N, w, P, ep, s);
    else rc = few ? launch_held<EPI, DOWN, 1>(x, N, w, P, ep, s) : launch_held<EPI, DOWN, 3>(x, N, w, P, ep, s);
    return true;
}
template int pairs_layer<EPI_NONE, false>(const float*, int64_t, int, const float*, int, const Epilogue&, void*, hipStream_t);
template int pairs_layer<EPI_GELU, false>(const float*, int64_t, int, const float*, int, const Epilogue&, void*, hipStream_t);
template int pairs_layer<EPI_RESIDUAL, false>(const float*, int64_t, int, const float*, int, const Epilogue&, void*, hipStream_t);
template int pairs_layer<EPI_NONE, true>(const float*, int64_t, int, const float*, int, const Epilogue&, void*, hipStream_t);
template int pairs_layer<EPI_SCALE, true>(const float*, int64_t, int, const float*, int, const Epilogue&, void*, hipStream_t);
template bool pairs_held<EPI_NONE, false>(const float*, int64_t, const float*, int, const Epilogue&, hipStream_t, int&);
template bool pairs_held<EPI_GELU, false>(const float*, int64_t, const float*, int, const Epilogue&, hipStream_t, int&);
template bool pairs_held<EPI_RESIDUAL, false>(const float*, int64_t, const float*, int, const Epilogue&, hipStream_t, int&);
template bool pairs_held<EPI_NONE, true>(const float*, int64_t, const float*, int, const Epilogue&, hipStream_t, int&);
template bool pairs_held<EPI_SCALE, true>(const float*, int64_t, const float*, int, const Epilogue&, hipStream_t, int&);

}  // namespace dense
}  // namespace sswin
