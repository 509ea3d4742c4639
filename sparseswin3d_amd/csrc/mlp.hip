// The feed-forward part of a block (sparse_swin/swin3d_base.py:700-706, 851-873) as one launch: both of its layers, the
// step between them and what follows the second one.
//   forward    g = GELU(x W1^T + b1), y = g W2^T + b2 + residual     (g and the derivative of GELU stored for the backward)
//   backward   du = (dy W2) * slope, dx = du W1                      (du stored for the weight gradients)
// Both are y = step(x A^T) B^T with A [hidden, D] and B [D, hidden]: A = W1, B = W2 forward, A = W2^T, B = W1^T backward.
//
// As two launches of dense.hip the hidden rows (4 D values a token) are written and read back between the layers and every
// launch is bound by that traffic; inference does not need them in memory at all.  Here a wavefront owns 32 tokens.  Products are
// formed transposed, z^T [hidden, tokens] = A x^T, so that an accumulator lane holds one token: with the rows of A permuted
// (hidden_of) its 16 values of a 32-wide hidden tile are two runs of eight neighbours, which is the operand of the second product
// y^T += B z^T in place.  No exchange between lanes, no round through LDS.  x stays in registers for the whole launch (96 channels:
// 24 registers, as two pieces of fp32 48), y accumulates in registers, A and B pass from L2 into LDS a step of 32 hidden
// channels at a time, the next step in flight, shared by the wavefronts of the workgroup.  What is stored or read per hidden value (g,
// slope, du) goes through a tile of LDS per wavefront, so that it is touched in runs of 64 or 128 bytes (16 bits straight from
// the accumulators, runs of 32 bytes: 225 000 rows fp16 48 channels 95 us, through the tile 69).
//
// fp32 operands are pairs of fp16 (Pairs of dense_operand.hpp).  A scale per row of x, found when the row is loaded, and per row of A and
// B, found by the launch that splits them; the hidden values' scale follows the largest of the token so far, and since a token's
// results lie in its own lanes, dropping it is a product a register.
// Small results are formed again (PAIRS_SMALL): hidden values where the wavefront's rows of x or any row of A have lost bits, which is
// known before the first step (225 700 rows, inference 178 -> 184 us; looked for in every step 190), values of y always.
//
// Microseconds, two launches (of three bf16 pieces) and one.  225 700 rows fp32 96 channels: forward 339 and 264, inference 296 and 184, backward
// 285 and 200 (with three pieces here 308, 227 and 245; traffic alone at copy rate 187 and 170 for the first and last).  Error against float64 (2-norms) of
// y 1.0e-7, three pieces 1.8e-7, of dx 1.9e-7 and 3.4e-7.  What bounds fp32 now: the stores of training, GELU on the vector units (about 26
// instructions of 45 a hidden value) and the products, of which two wavefronts a SIMD cover two thirds with each other.
// fp16 48 channels, 225 000 rows: 89 and 69, 55 and 43 (55 and 38).  bf16 96 channels, inference, 112 700 rows: 65 and 45 (13; GELU on
// the vector units 21).
#include <algorithm>
#include <initializer_list>
#include <type_traits>

#include "dense_epilogue.hpp"
#include "dense_operand.hpp"
#include "mfma_block.hpp"
#include "sswin_common.hpp"

namespace sswin {
namespace dense {

struct MlpArgs {
    const void* x;             // [N, D]
    int64_t N;
    int hidden;
    const uint16_t* a;         // [planes][hidden, D]
    const uint16_t* b;         // [planes][D, hidden]
    const int *ea, *eb;        // fp32: exponents of the scales of their rows
    const float *wa, *wb;      // fp32: what the pieces are of, forward [hidden, D] and [D, hidden], backward turned
    const void* bias_a;        // [hidden] or null
    const void* bias_b;        // [D] or null
    const void* factor;        // backward: slope [N, hidden]
    const void* residual;      // forward: [N, D] of y's type, or null
    void* h;                   // g or du [N, hidden]
    void* slope;               // forward: [N, hidden]
    void* y;                   // [N, D]
    int64_t full;              // workgroups whose wavefronts all have 32 tokens; in those behind them the first `some` have
    int some;
};

constexpr int MLP_LDS = 160 * 1024;
enum { MLP_INFER, MLP_TRAIN, MLP_BACKWARD };

// row of the hidden tile (of an output tile) that is put into row i of the operand: accumulator register 8 s + e of half h is
// then row 16 s + 8 h + e
__device__ __forceinline__ int hidden_of(int i) { return (i & 0x13) | (i & 4) << 1 | (i & 8) >> 1; }

template <typename T> constexpr int MLP_PL = sizeof(T) == 4 ? 2 : 1;     // planes of an operand

// a wavefront's rows as operands; the exponent of the scale of the lane's row (fp32), and whether the pieces lose bits of its part of it
template <typename T, int KS> __device__ __forceinline__ int load_rows(const T* p, u32x4 (&x)[KS][MLP_PL<T>], bool& lost) {
    if constexpr (sizeof(T) == 4) {
        float v[KS][8], m = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const f32x4 lo = *reinterpret_cast<const f32x4*>(p + ks * 16), hi = *reinterpret_cast<const f32x4*>(p + ks * 16 + 4);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[ks][e] = e < 4 ? lo[e] : hi[e - 4];
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) m = fmaxf(m, largest(v[ks]));
        const int e = pairs_scale(exponent_above(largest_of_halves(m)));
        const float scale = power_of_two(e);
        uint32_t least = 0xffffffffu;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) least = least_nonzero(v[ks], least);
        lost = pairs_lose(least, scale);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) split_pairs(v[ks], scale, x[ks]);
        return e;
    } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) x[ks][0] = *reinterpret_cast<const u32x4*>(p + ks * 16);
        return 0;
    }
}

// 32 hidden values (or columns of y) of a wavefront's 32 tokens in LDS, so that memory is touched in runs of a row: rows of ROW
// 16-byte pieces, the pieces of a row exchanged by its number.  Own side: the lane's token; memory side: slots in their order.
template <typename T> struct HiddenTile {
    static constexpr int VALUES = 16 / (int)sizeof(T), ROW = 32 / VALUES, PIECES = 32 * ROW, MOVES = PIECES / 64, STEP_ROWS = 64 / ROW;
    static __device__ __forceinline__ int slot(int r, int piece) { return r * ROW + (piece ^ (ROW == 8 ? r & 7 : r >> 1 & 3)); }
    // row and first column of this lane's slot of the first 64; the same column in the others
    static __device__ __forceinline__ int mem_row() { return (threadIdx.x & 63) / ROW; }
    static __device__ __forceinline__ int mem_col() {
        const int r = mem_row(), s = (threadIdx.x & 63) % ROW;
        return (slot(r, s) - r * ROW) * VALUES;
    }
    // the values 16 s + 8 half .. + 7 of the own token
    static __device__ __forceinline__ void put(u32x4* tile, int s, const float (&v)[8]) {
        const int half = (threadIdx.x & 63) >> 5, l32 = threadIdx.x & 31;
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
                tile[slot(l32, s * 4 + half * 2 + h)] = __builtin_bit_cast(u32x4, f32x4{v[4 * h], v[4 * h + 1], v[4 * h + 2], v[4 * h + 3]});
        } else {
            u32x4 p[1];
            planes_of<T>(v, p);
            tile[slot(l32, s * 2 + half)] = p[0];
        }
    }
    static __device__ __forceinline__ void get(const u32x4* tile, int s, float (&v)[8]) {
        const int half = (threadIdx.x & 63) >> 5, l32 = threadIdx.x & 31;
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f32x4 p = __builtin_bit_cast(f32x4, tile[slot(l32, s * 4 + half * 2 + h)]);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[4 * h + e] = p[e];
            }
        } else {
            const Vec8<T> p = __builtin_bit_cast(Vec8<T>, tile[slot(l32, s * 2 + half)]);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = to_acc(p.q[e / 4].v[e % 4]);
        }
    }
};

// the step between the layers on eight hidden values
template <typename T, int MODE>
__device__ __forceinline__ void between(const f32x16& z, int s, const float* bias, const u32x4* tile, float (&v)[8], float (&u)[8]) {
    if constexpr (MODE == MLP_BACKWARD) {
        HiddenTile<T>::get(tile, s, u);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = z[s * 8 + e] * u[e];
    } else {
        const f32x4* const b8 = reinterpret_cast<const f32x4*>(bias + s * 16 + ((threadIdx.x & 63) >> 5) * 8);
        const f32x4 b[2] = {b8[0], b8[1]};
#pragma unroll
        for (int e = 0; e < 8; ++e) gelu_and_slope<sizeof(T) == 4>(z[s * 8 + e] + b[e / 4][e % 4], v[e], u[e]);
    }
}

// y of a wavefront's 32 tokens from row0 on, 32 columns at a time through a tile of fp32 values
template <typename TO, int D, int MODE>
__device__ __forceinline__ void store_y(const MlpArgs& g, const f32x16 (&y)[(D + 31) / 32], int64_t row0, const float* bias, u32x4* tile) {
    using Y = HiddenTile<float>;
#pragma unroll
    for (int j = 0; j < (D + 31) / 32; ++j) {
        const int col = j * 32 + Y::mem_col();
        const bool in = D % 32 == 0 || col < D;
        const int64_t at = (row0 + Y::mem_row()) * D + col;
        Vec4<TO> r[4];
        if (MODE != MLP_BACKWARD && g.residual && in)
#pragma unroll
            for (int i = 0; i < 4; ++i) r[i] = *reinterpret_cast<const Vec4<TO>*>(static_cast<const TO*>(g.residual) + at + i * 8 * D);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = y[j][s * 8 + e];
            Y::put(tile, s, v);
        }
        __builtin_amdgcn_wave_barrier();
        if (in)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4 v = __builtin_bit_cast(f32x4, tile[i * 64 + (threadIdx.x & 63)]);
                float o[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[e] = v[e];
                    if constexpr (MODE != MLP_BACKWARD) {
                        o[e] += bias[col + e];
                        if (g.residual) o[e] += to_acc(r[i].v[e]);
                    }
                }
                *reinterpret_cast<Vec4<TO>*>(static_cast<TO*>(g.y) + at + i * 8 * D) = pack4<TO>(o);
            }
    }
}
template <typename T> __device__ __forceinline__ void stage_biases(const MlpArgs& g, int D, float* bias) {
    for (int e = threadIdx.x; e < g.hidden; e += (int)blockDim.x) bias[e] = g.bias_a ? to_acc(static_cast<const T*>(g.bias_a)[e]) : 0.f;
    for (int e = threadIdx.x; e < D; e += (int)blockDim.x) bias[g.hidden + e] = g.bias_b ? to_acc(static_cast<const T*>(g.bias_b)[e]) : 0.f;
}
// fp32: y where the pieces left NaN, again in plain fp32 as in dense.hip (plain_products), and the hidden values before it with what is
// stored of them.  A hidden value that came out NaN makes every y of its token NaN, so y alone tells, once a launch.  Inference has
// no hidden values in memory and forms all of these tokens again; so does training for y, for the same bits.
template <int D, int MODE> __device__ __forceinline__ void plain_rows(const MlpArgs& g, int64_t row0, const float* bias, u32x4* tile, f32x16 (&y)[(D + 31) / 32]) {
    constexpr int CT = (D + 31) / 32;
    using H = HiddenTile<float>;
    const int half = (threadIdx.x & 63) >> 5, l32 = threadIdx.x & 31;
    const int64_t row = row0 + l32;
    f32x16 p[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) p[j] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    wait_copies<0>();                                                    // the stores of this wavefront, read here
#pragma unroll 1
    for (int k0 = 0; k0 < g.hidden; k0 += 32) {
#pragma unroll 1
        for (int c = 0; c < 4; ++c) {
            const int k = k0 + half * 16 + c * 4;
            f32x4* const stored = reinterpret_cast<f32x4*>(static_cast<float*>(g.h) + row * g.hidden + k);
            f32x4 v;
            if (MODE != MLP_INFER) v = *stored;
            const bool nan = MODE != MLP_INFER && nan_among(v);
            if (MODE != MLP_BACKWARD || nan) {
                const float* const x = static_cast<const float*>(g.x) + row * D;
                f32x4 u;
                if constexpr (MODE == MLP_BACKWARD) {
                    v = plain_products(x, 1, g.wa + k, g.hidden, 1, D);
                    u = *reinterpret_cast<const f32x4*>(static_cast<const float*>(g.factor) + row * g.hidden + k);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] *= u[e];
                } else {
                    v = plain_products(x, 1, g.wa + (int64_t)k * D, 1, D, D);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float act, slope;
                        gelu_and_slope<true>(v[e] + bias[k + e], act, slope);
                        v[e] = act, u[e] = slope;
                    }
                }
                if (nan) *stored = v;
                if (MODE == MLP_TRAIN && nan) *reinterpret_cast<f32x4*>(static_cast<float*>(g.slope) + row * g.hidden + k) = u;
            }
            tile[H::slot(l32, half * 4 + c)] = __builtin_bit_cast(u32x4, v);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (int c = 0; c < 8; ++c) {
            const f32x4 v = __builtin_bit_cast(f32x4, tile[H::slot(l32, c)]);
#pragma unroll 1
            for (int e = 0; e < 4; ++e) {
                const int k = k0 + c * 4 + e;
                const float f = e == 0 ? v[0] : e == 1 ? v[1] : e == 2 ? v[2] : v[3];
#pragma unroll
                for (int j = 0; j < CT; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int col = j * 32 + r / 8 * 16 + half * 8 + r % 8;
                        p[j][r] = fmaf(f, MODE == MLP_BACKWARD ? g.wb[(int64_t)k * D + col] : g.wb[(int64_t)col * g.hidden + k], p[j][r]);
                    }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) y[j][r] = y[j][r] == y[j][r] ? y[j][r] : p[j][r];
}

// The small ones among a tile's values (PAIRS_SMALL; register 8 s + e of half h is row 16 s + 8 h + e, the lane's token column), of scales ex and exps, from
// product(token, row); true: they are many, and marked with NaN, which makes their tokens those of plain_rows.
template <typename F> __device__ __forceinline__ bool small_again(f32x16& z, int ex, const int* exps, F product) {
    const int lane = threadIdx.x & 63;
    uint32_t mask = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int ew = exps[r / 8 * 16 + (lane >> 5) * 8 + r % 8];
        if (ew <= PAIRS_MOST_SCALE && fabsf(__builtin_amdgcn_ldexpf(z[r], ex + ew)) < PAIRS_SMALL) mask |= 1u << r;
    }
    if (ex > PAIRS_MOST_SCALE) mask = 0;
    if (!__any(mask)) return false;
    if (many_small(mask)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) z[r] = mask >> r & 1 ? NAN : z[r];
        return true;
    }
    for_each_small(mask, [&](int owner, int bit) {
        const float v = product(owner & 31, bit / 8 * 16 + (owner >> 5) * 8 + bit % 8);
#pragma unroll
        for (int r = 0; r < 16; ++r) z[r] = lane == owner && bit == r ? v : z[r];
    });
    return false;
}
// y of one token and column in plain fp32, without its bias, by the wavefront: from du in memory, or from hidden values formed again
template <int D, int MODE> __device__ __forceinline__ float one_output(const MlpArgs& g, int64_t row, int col, const float* bias) {
    const float* const w = g.wb + (MODE == MLP_BACKWARD ? col : (int64_t)col * g.hidden);
    if constexpr (MODE == MLP_BACKWARD) return wave_product(static_cast<const float*>(g.h) + row * g.hidden, w, D, g.hidden);
    const float* const x = static_cast<const float*>(g.x) + row * D;
    float y = 0.f;
#pragma unroll 1
    for (int k = threadIdx.x & 63; k < g.hidden; k += 64) {
        const f32x4* const a = reinterpret_cast<const f32x4*>(g.wa + (int64_t)k * D);
        float z = 0.f, act, slope;
#pragma unroll 4
        for (int i = 0; i < D / 4; ++i) {
            const f32x4 v = a[i];
#pragma unroll
            for (int e = 0; e < 4; ++e) z = fmaf(x[i * 4 + e], v[e], z);
        }
        gelu_and_slope<true>(z + bias[k], act, slope);
        y = fmaf(act, w[k], y);
    }
    return wave_sum(y);
}

// A step is 32 hidden channels.  The wait for the next step's A and B leaves the stores of this step in flight; it counts them, so they
// are inline assembly.
template <typename T, int D, int MODE, int WAVES> struct MlpLds {
    static constexpr int PIECES = MLP_PL<T> * (D / 16 + 2 * ((D + 31) / 32));   // of 64 x 16 bytes, a step's A and B
    // of 16 bytes, a wavefront's tiles: two of hidden values, at least one of y.  Inference: y leaves through the place of A and B
    // where it is large enough
    static constexpr bool SHARED = MODE == MLP_INFER && WAVES * 256 <= 2 * PIECES * 64;
    static constexpr int OWN = SHARED ? 0 : std::max(256, 2 * HiddenTile<T>::PIECES);
    static constexpr int PER_CHANNEL = sizeof(T) == 4 ? 2 : 1;           // its bias, and fp32 the exponent of its scale
    static constexpr int FLAGS = sizeof(T) == 4 ? (WAVES + 3) / 4 : 0;   // 16-byte pieces with one a wavefront
    static size_t bytes(int hidden) { return (size_t)2 * PIECES * 1024 + (size_t)(hidden + D) * 4 * PER_CHANNEL + FLAGS * 16 + (size_t)WAVES * OWN * 16; }
};
template <typename T, typename TO, int D, int MODE, int WAVES, int OCC>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void mlp_kernel(MlpArgs g) {
    using L = MlpLds<T, D, MODE, WAVES>;
    using H = HiddenTile<T>;
    constexpr int PL = MLP_PL<T>, KS = D / 16, CT = (D + 31) / 32, PA = KS * PL, PIECES = L::PIECES;
    constexpr int STORES = MODE == MLP_INFER ? 0 : MODE == MLP_TRAIN ? 2 * H::MOVES : H::MOVES;
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    float* const bias = reinterpret_cast<float*>(lds + 2 * PIECES * 64); // [hidden] and [D]
    int* const exps = reinterpret_cast<int*>(bias + g.hidden + D);       // fp32: the same
    int* const lost_ab = exps + g.hidden + D;                            // fp32: whether a wavefront has seen rows of A (1) and B (2) that lose bits
    u32x4* const tiles = L::SHARED ? lds + wave * 256 : lds + 2 * PIECES * 64 + (g.hidden + D) * L::PER_CHANNEL / 4 + L::FLAGS + wave * L::OWN;
    const int64_t behind = (int64_t)blockIdx.x - g.full, row0 = tile_row(behind < 0 ? (int64_t)blockIdx.x * WAVES + wave : g.full * WAVES + behind * g.some + wave, g.N);
    const int64_t plane = (int64_t)g.hidden * D;
    const uint32_t lane_a = (uint32_t)(hidden_of(l32) * D + half * 8);
    auto request = [&](int step) {
        const uint32_t to = lds_address(lds) + (uint32_t)(step & 1) * PIECES * 1024;
#pragma unroll
        for (int q = 0; q < (PIECES + WAVES - 1) / WAVES; ++q) {
            const int p = q * WAVES + wave, r = p - PA;                  // uniform in the wavefront
            if (PIECES % WAVES != 0 && p >= PIECES) break;
            const uint16_t* from;
            if (p < PA) from = g.a + p % PL * plane + (int64_t)step * 32 * D + p / PL * 16 + lane_a;
            else from = g.b + r % PL * plane + (int64_t)min(r / PL % CT * 32 + hidden_of(l32), D - 1) * g.hidden + step * 32 + r / (PL * CT) * 16 + half * 8;
            copy_to_lds(from, to + (uint32_t)p * 1024);
        }
    };
    const int steps = g.hidden / 32;
    request(0);
    if constexpr (MODE != MLP_BACKWARD) stage_biases<T>(g, D, bias);
    if constexpr (PL == 2) {
        bool seen_a = false, seen_b = false;
        for (int c = threadIdx.x; c < g.hidden + D; c += WAVES * 64) {
            const int e = c < g.hidden ? g.ea[c] : g.eb[c - g.hidden], cut = e >= PAIRS_LOST / 2 ? PAIRS_LOST : 0;
            exps[c] = e - cut;
            seen_a |= cut && c < g.hidden, seen_b |= cut && c >= g.hidden;
        }
        lost_ab[wave] = (__any(seen_a) ? 1 : 0) | (__any(seen_b) ? 2 : 0);
    }
    if (behind >= 0 && wave >= g.some) {                                 // without tokens: only brings A and B
        wait_copies<0>();
        if constexpr (PL == 2) block_barrier();
        for (int step = 0; step < steps; ++step) {
            block_barrier();
            if (step + 1 < steps) request(step + 1);
            wait_copies<0>();
        }
        if constexpr (L::SHARED) block_barrier();
        return;
    }
    u32x4 x[KS][PL];
    bool lost = false;
    const int ex = load_rows<T, KS>(static_cast<const T*>(g.x) + (row0 + l32) * D + half * 8, x, lost);
    const int64_t mem = (row0 + H::mem_row()) * g.hidden + H::mem_col();
    auto load_tile = [&](int step) {                                     // of slope
#pragma unroll
        for (int i = 0; i < H::MOVES; ++i)
            copy_to_lds(static_cast<const T*>(g.factor) + mem + (int64_t)i * H::STEP_ROWS * g.hidden + step * 32,
                        lds_address(tiles + (step & 1) * H::PIECES + i * 64));
    };
    auto store_tile = [&](const u32x4* tile, void* to, int step) {
        u32x4 v[H::MOVES];
#pragma unroll
        for (int i = 0; i < H::MOVES; ++i) v[i] = tile[i * 64 + lane];
#pragma unroll
        for (int i = 0; i < H::MOVES; ++i) store_counted(static_cast<T*>(to) + mem + (int64_t)i * H::STEP_ROWS * g.hidden + step * 32, v[i]);
    };
    f32x16 y[CT], y_low[PL == 2 ? CT : 1];
#pragma unroll
    for (int j = 0; j < CT; ++j) y[j] = y_low[PL == 2 ? j : 0] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    int eh = PAIRS_ZEROS_SO_FAR;                                         // fp32: exponent of the scale of the row's hidden values
    float hidden_scale = 0.f;
    if constexpr (MODE == MLP_BACKWARD) load_tile(0);
    wait_copies<0>();
    int ab = 0;
    if constexpr (PL == 2) {
        block_barrier();
#pragma unroll
        for (int w = 0; w < WAVES; ++w) ab |= lost_ab[w];
        lost = __any(lost || (ab & 1));                                  // results of operands that lose no bits may be small
    }
    float least_hidden = INFINITY;
    if (PL == 2 && wave < WAVES / 2) __builtin_amdgcn_s_setprio(1);      // the two wavefronts of a SIMD at different places of a step
    // twice in the code, since a branch for small hidden values in the loop costs 3 % where there are none
    auto run = [&](auto small) {
        for (int step = 0; step < steps; ++step) {
            block_barrier();                                                 // this buffer is there, the other one is free
            if (step + 1 < steps) {
                request(step + 1);
                if constexpr (MODE == MLP_BACKWARD) load_tile(step + 1);
            }
            u32x4* const tile = tiles + (MODE == MLP_BACKWARD ? (step & 1) * H::PIECES : 0);   // du takes the place of its slope
            const u32x4* const pieces = lds + (step & 1) * PIECES * 64 + lane;
            // z^T: the pieces of A are read a slice of 16 channels ahead of its products
            f32x16 z = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0}, z_low = z;
            u32x4 a[2][PL];
#pragma unroll
            for (int q = 0; q < PL; ++q) a[0][q] = pieces[q * 64];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                if (ks + 1 < KS)
#pragma unroll
                    for (int q = 0; q < PL; ++q) a[(ks + 1) & 1][q] = pieces[((ks + 1) * PL + q) * 64];
                if constexpr (PL == 2) {
                    z_low = Pairs::mfma(a[ks & 1][1], x[ks][0], z_low);
                    z = Pairs::mfma(a[ks & 1][0], x[ks][0], z);
                    z_low = Pairs::mfma(a[ks & 1][0], x[ks][1], z_low);
                } else {
                    z = Op<T>::mfma(a[ks & 1][0], x[ks][0], z);
                }
                __builtin_amdgcn_sched_group_barrier(0x100, PL, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, PL == 2 ? 3 : 1, 0);
            }
            if constexpr (PL == 2) {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const int4* const e8 = reinterpret_cast<const int4*>(exps + step * 32 + s * 16 + half * 8);
                    const int4 lo = e8[0], hi = e8[1];
                    const int ew[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) z[s * 8 + e] = __builtin_amdgcn_ldexpf(fmaf(z_low[s * 8 + e], Pairs::LOW, z[s * 8 + e]), -(ex + ew[e]));
                }
                if constexpr (decltype(small)::value)
                    small_again(z, ex, exps + step * 32, [&](int l, int c) {
                        const int k = step * 32 + c;
                        return wave_product(static_cast<const float*>(g.x) + (row0 + l) * D, g.wa + (MODE == MLP_BACKWARD ? k : (int64_t)k * D),
                                            MODE == MLP_BACKWARD ? g.hidden : 1, D);
                    });
            }
            auto step_between = [&](int s, float (&v)[8]) {
                float u[8];
                between<T, MODE>(z, s, bias + step * 32, tile, v, u);
                if constexpr (MODE != MLP_INFER) H::put(tile, s, v);
                if constexpr (MODE == MLP_TRAIN) H::put(tile + H::PIECES, s, u);
            };
            auto second_layer = [&](int s, const u32x4 (&h)[PL]) {
                u32x4 w[2][PL];
                auto read = [&](int j) {
#pragma unroll
                    for (int q = 0; q < PL; ++q) w[j & 1][q] = pieces[(PA + (s * CT + j) * PL + q) * 64];
                };
                read(0);
#pragma unroll
                for (int j = 0; j < CT; ++j) {
                    if (j + 1 < CT) read(j + 1);
                    if constexpr (PL == 2) {
                        y_low[j] = Pairs::mfma(w[j & 1][1], h[0], y_low[j]);
                        y[j] = Pairs::mfma(w[j & 1][0], h[0], y[j]);
                        y_low[j] = Pairs::mfma(w[j & 1][0], h[1], y_low[j]);
                    } else {
                        y[j] = Op<T>::mfma(w[j & 1][0], h[0], y[j]);
                    }
                }
            };
            u32x4 h[PL];
            if constexpr (PL == 2) {
                float v[2][8];
                step_between(0, v[0]);
                step_between(1, v[1]);
                // the scale follows the largest value seen: where a step's would leave fp16's range it drops, and the sums with it
                const int above = exponent_above(largest_of_halves(fmaxf(largest(v[0]), largest(v[1]))));
                if constexpr (MODE == MLP_INFER)
#pragma unroll
                    for (int e = 0; e < 16; ++e) least_hidden = least_size(least_hidden, v[e / 8][e % 8]);
                if (__any(above + eh > 15)) {
                    const int now = pairs_scale_after(above, eh);
                    const float factor = power_of_two(now - eh);
                    eh = now, hidden_scale = power_of_two(min(now, PAIRS_MOST_SCALE));
#pragma unroll
                    for (int j = 0; j < CT; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r) y[j][r] *= factor, y_low[j][r] *= factor;
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    split_pairs(v[s], hidden_scale, h);
                    second_layer(s, h);
                }
            } else {
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    float v[8];
                    step_between(s, v);
                    planes_of<T>(v, h);
                    second_layer(s, h);
                }
            }
            if constexpr (MODE != MLP_INFER) {
                __builtin_amdgcn_wave_barrier();
                store_tile(tile, g.h, step);
                if constexpr (MODE == MLP_TRAIN) store_tile(tile + H::PIECES, g.slope, step);
                __builtin_amdgcn_wave_barrier();
            }
            if (step + 1 < steps) wait_copies<STORES>();                     // all but the stores of this step
        }
    };
    if (lost) run(std::true_type());
    else run(std::false_type());
    if constexpr (L::SHARED) block_barrier();                    // A and B have been read
    if constexpr (PL == 2) {
        float least = INFINITY;
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int ew = exps[g.hidden + j * 32 + r / 8 * 16 + half * 8 + r % 8];
                const float t = fmaf(y_low[j][r], Pairs::LOW, y[j][r]);
                least = least_size(least, t);
                y[j][r] = __builtin_amdgcn_ldexpf(t, -(eh + ew));
            }
        bool small = nan_or_small(least, eh);
        if (__any(small)) {
            wait_copies<0>();                                            // the hidden values stored by this wavefront are read
            // In inference a value of y takes its hidden values again, 13 us: only where one of them, or of B, has lost bits.  The same in training,
            // so that both give the same bits.
            if constexpr (MODE != MLP_BACKWARD) {
                if constexpr (MODE == MLP_INFER) least_hidden = fminf(least_hidden, __shfl_xor(least_hidden, 32, 64));      // the token's others
                else
                    for_each_small(small ? 1u : 0u, [&](int owner, int) {
                        const float* const h = static_cast<const float*>(g.h) + (row0 + (owner & 31)) * g.hidden;
                        float m = INFINITY;
                        for (int k = lane; k < g.hidden; k += 64) m = least_size(m, h[k]);
                        m = wave_least(m);
                        if (lane == owner) least_hidden = m;
                    });
                small = small && ((ab & 2) || __builtin_amdgcn_ldexpf(least_hidden, eh) < 0x1p-13f);
            }
            bool nan = __any(least != least);
#pragma unroll
            for (int j = 0; j < CT; ++j)
                nan |= small_again(y[j], small ? eh : PAIRS_ZEROS, exps + g.hidden + j * 32,
                                   [&](int l, int c) { return one_output<D, MODE>(g, row0 + l, j * 32 + c, bias); });
            if (nan) plain_rows<D, MODE>(g, row0, bias, tiles, y);
        }
    }
    store_y<TO, D, MODE>(g, y, row0, bias + g.hidden, tiles);
}

// ------------------------------------------------------------------------------------------
// y [N, P] = x [N, D] W^T + b for 16-bit rows and few input channels, the first half of the kernel above: a wavefront keeps its
// 32 tokens of x in registers and forms y^T 32 columns at a time, so that a row of x is read once and by one workgroup (the tiles of
// dense.hip read it once per 96 columns of y, and start anew for each).  Bound by the stores of y.  W passes through LDS a step of 32 columns at a time.
// ------------------------------------------------------------------------------------------
// CT tiles of 32 columns a step; OWN: 16-byte pieces of a wavefront's 32 x 32 CT results
template <int D, int CT, int WAVES> struct RowsOnceLds {
    static constexpr int PIECES = D / 16 * CT, OWN = CT * 128;
    static size_t bytes(int P) { return (size_t)2 * PIECES * 1024 + (size_t)WAVES * OWN * 16 + (size_t)(P + CT * 32 - 1) / (CT * 32) * CT * 128; }
};
template <typename T, int D, int CT, int WAVES, int OCC>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void rows_once_kernel(const T* __restrict__ x, int64_t N,
                                                                                                     const T* __restrict__ w, const T* __restrict__ b, int P,
                                                                                                     T* __restrict__ y) {
    using L = RowsOnceLds<D, CT, WAVES>;
    using H = HiddenTile<typename std::conditional<CT == 2, float, T>::type>;                             // rows of 64 or 128 bytes
    constexpr int KS = D / 16, PIECES = L::PIECES;
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
    u32x4* const tile = lds + 2 * PIECES * 64 + wave * L::OWN;
    float* const bias = reinterpret_cast<float*>(lds + 2 * PIECES * 64 + WAVES * L::OWN);
    const int64_t row0 = tile_row((int64_t)blockIdx.x * WAVES + wave, N);
    const int steps = (P + CT * 32 - 1) / (CT * 32);
    auto request = [&](int step) {
#pragma unroll
        for (int q = 0; q < (PIECES + WAVES - 1) / WAVES; ++q) {
            const int p = q * WAVES + wave;                              // uniform in the wavefront
            if (PIECES % WAVES != 0 && p >= PIECES) break;
            copy_to_lds(w + (int64_t)min((step * CT + p / KS) * 32 + hidden_of(l32), P - 1) * D + p % KS * 16 + half * 8,
                        lds_address(lds) + (uint32_t)((step & 1) * PIECES + p) * 1024);
        }
    };
    request(0);
    for (int e = threadIdx.x; e < steps * CT * 32; e += WAVES * 64) bias[e] = b && e < P ? to_acc(b[e]) : 0.f;
    u32x4 rows[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) rows[ks] = *reinterpret_cast<const u32x4*>(x + (row0 + l32) * D + ks * 16 + half * 8);
    const int col = H::mem_col() * (CT == 2 ? 2 : 1);                    // pieces of eight values either way
    const int64_t mem = (row0 + H::mem_row()) * P + col;
    wait_copies<0>();
    for (int step = 0; step < steps; ++step) {
        block_barrier();                                                 // this buffer is there, the other one is free
        if (step + 1 < steps) request(step + 1);
        const u32x4* const pieces = lds + (step & 1) * PIECES * 64 + lane;
        f32x16 z[CT];
#pragma unroll
        for (int t = 0; t < CT; ++t) {
            z[t] = f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) z[t] = Op<T>::mfma(pieces[(t * KS + ks) * 64], rows[ks], z[t]);
        }
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const f32x4* const b8 = reinterpret_cast<const f32x4*>(bias + (step * CT + t) * 32 + s * 16 + half * 8);
                const f32x4 b01[2] = {b8[0], b8[1]};
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = z[t][s * 8 + e] + b01[e / 4][e % 4];
                u32x4 p[1];
                planes_of<T>(v, p);
                tile[H::slot(l32, t * 4 + s * 2 + half)] = p[0];
            }
        __builtin_amdgcn_wave_barrier();
        u32x4 out[H::MOVES];
#pragma unroll
        for (int i = 0; i < H::MOVES; ++i) out[i] = tile[i * 64 + lane];
        if (step * CT * 32 + col < P)                                    // 16 columns at least: the stores are counted
#pragma unroll
            for (int i = 0; i < H::MOVES; ++i) store_counted(y + mem + (int64_t)i * H::STEP_ROWS * P + step * CT * 32, out[i]);
        __builtin_amdgcn_wave_barrier();
        if (step + 1 < steps) wait_copies<H::MOVES>();                   // all but the stores of this step
    }
}
template <typename K> static int allow_all_lds(K* k) {
    SSWIN_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, MLP_LDS));
    return 0;
}
template <typename T, int D, int CT, int WAVES, int OCC> static int launch_rows_once(const T* x, int64_t N, const T* w, const T* b, int P, T* y, hipStream_t s) {
    auto* k = rows_once_kernel<T, D, CT, WAVES, OCC>;
    static const int configured = allow_all_lds(k);
    if (configured) return configured;
    hipLaunchKernelGGL(k, dim3((unsigned)((N + WAVES * 32 - 1) / (WAVES * 32))), dim3(WAVES * 64), (RowsOnceLds<D, CT, WAVES>::bytes(P)), s, x, N, w, b, P, y);
    return launch_ok("rows once");
}
// The rows from which this is ahead of the tiles of dense.hip (microseconds, tiles and here).  bf16 96 -> 288: 8000 rows 7.0 and 8.0,
// 16 000 12.0 and 8.8, 112 700 23.1 and 17.5, 445 000 108 and 83 (67 at copy rate).  fp16 48 -> 144: 4000 4.0 and 4.6, 8000 4.9 and 4.8,
// 225 000 25.0 and 19.1 (17).  bf16 192 -> 576: 37 000 22.7 and 24.2, 50 000 28.5 and 25.3, 147 000 64.7 and 55.2 (44): with fewer rows a
// compute unit has too few workgroups to hide where each one starts.  With GELU 192 -> 768 loses up to 100 000 rows.
bool rows_once_takes(int64_t N, int D, int P) {
    return N < (1ll << 31) && P <= 2048 && ((D == 48 && N >= 8000) || (D == 96 && N >= 16000) || (D == 192 && N >= 50000));
}
// 64 columns a step (runs of 128 bytes), with 192 channels 32, for the place their pieces of W take; 445 000 rows 96 -> 288: 92 us with 32
template <typename T> int rows_once(const T* x, int64_t N, int D, const T* w, const T* b, int P, T* y, hipStream_t s) {
    if (D == 48) return launch_rows_once<T, 48, 2, 4, 5>(x, N, w, b, P, y, s);
    if (D == 96) return launch_rows_once<T, 96, 2, 8, 4>(x, N, w, b, P, y, s);
    return launch_rows_once<T, 192, 1, 8, 4>(x, N, w, b, P, y, s);
}
template int rows_once<__half>(const __half*, int64_t, int, const __half*, const __half*, int, __half*, hipStream_t);
template int rows_once<__hip_bfloat16>(const __hip_bfloat16*, int64_t, int, const __hip_bfloat16*, const __hip_bfloat16*, int, __hip_bfloat16*, hipStream_t);

// A and B of the backward, weights turned, 16 bit: a thread per pair of neighbours of a row
template <typename T>
__global__ __launch_bounds__(256) void mlp_weights_kernel(const T* __restrict__ wa, const T* __restrict__ wb, int D, int hidden, uint16_t* __restrict__ a,
                                                          uint16_t* __restrict__ b) {
    const int64_t pairs = (int64_t)D * hidden / 2, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= 2 * pairs) return;
    const bool second = i >= pairs;
    const int64_t e = (second ? i - pairs : i) * 2;
    const int cols = second ? hidden : D, rows = second ? D : hidden;    // of the result
    const int64_t r = e / cols, c = e % cols;
    const T* w = second ? wb : wa;
    const T v0 = w[c * rows + r], v1 = w[(c + 1) * rows + r];
    *reinterpret_cast<uint32_t*>((second ? b : a) + e) = (uint32_t)__builtin_bit_cast(uint16_t, v0) | (uint32_t)__builtin_bit_cast(uint16_t, v1) << 16;
}
// fp32: the pieces of both, and the exponents of their rows' scales; a workgroup per 32 rows
template <bool TURNED>
__global__ __launch_bounds__(512) void mlp_pairs_kernel(const float* __restrict__ wa, const float* __restrict__ wb, int D, int hidden, uint16_t* __restrict__ a,
                                                        uint16_t* __restrict__ b, int* __restrict__ ea, int* __restrict__ eb) {
    const bool second = (int)blockIdx.x >= hidden / 32;
    const int tile = second ? (int)blockIdx.x - hidden / 32 : (int)blockIdx.x, rows = second ? D : hidden, cols = second ? hidden : D;
    uint16_t* const to = second ? b : a;
    const int e = pairs_of_columns<TURNED, 8, true>(second ? wb : wa, cols, rows, tile, [&](int row, int ks, int half, const u32x4 (&p)[2]) {
#pragma unroll
        for (int q = 0; q < 2; ++q) *reinterpret_cast<u32x4*>(to + (int64_t)q * D * hidden + (int64_t)row * cols + ks * 16 + half * 8) = p[q];
    });
    if (threadIdx.x < 32) (second ? eb : ea)[tile * 32 + threadIdx.x] = e;
}

template <typename T, typename TO, int D, int MODE, int WAVES, int OCC> static int launch_mlp_as(MlpArgs g, hipStream_t s) {
    auto* k = mlp_kernel<T, TO, D, MODE, WAVES, OCC>;
    static const int configured = allow_all_lds(k);
    if (configured) return configured;
    // One workgroup of 8 wavefronts fills a compute unit: the tokens behind the last full round are dealt to all of them, so that fewer
    // wavefronts share a SIMD there.  (Smaller workgroups need no rule.)
    const int64_t tiles = (g.N + 31) / 32, cus = device_cus();
    g.full = WAVES == 8 ? tiles / (WAVES * cus) * cus : tiles / WAVES;
    const int64_t rest = tiles - g.full * WAVES;
    g.some = WAVES == 8 ? (int)((rest + cus - 1) / cus) : WAVES;
    const int64_t blocks = g.full + (rest ? (rest + g.some - 1) / g.some : 0);
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(WAVES * 64), (MlpLds<T, D, MODE, WAVES>::bytes(g.hidden)), s, g);
    return launch_ok("mlp");
}
template <typename T, typename TO, int MODE> static int launch_mlp(const MlpArgs& g, int D, hipStream_t s) {
    // wavefronts per SIMD: what the registers allow without spilling
    if constexpr (std::is_same<T, float>::value) return launch_mlp_as<T, TO, 96, MODE, 8, 2>(g, s);
    else if (D == 48) return launch_mlp_as<T, TO, 48, MODE, 4, 4>(g, s);
    else return launch_mlp_as<T, TO, 96, MODE, 4, MODE == MLP_INFER ? 4 : 3>(g, s);
}

// fp32: two planes of A, two of B, then the exponents of their rows
template <typename T> static int launch_weights(MlpArgs& g, const void* wa, const void* wb, bool turned, int D, int hidden, void* ws, hipStream_t s) {
    uint16_t *a = static_cast<uint16_t*>(ws), *b = a + (size_t)MLP_PL<T> * D * hidden;
    g.a = a, g.b = b;
    if constexpr (sizeof(T) == 4) {
        int *ea = reinterpret_cast<int*>(b + (size_t)2 * D * hidden), *eb = ea + hidden;
        g.ea = ea, g.eb = eb;
        const dim3 grid((unsigned)((hidden + D) / 32));
        auto* k = turned ? mlp_pairs_kernel<true> : mlp_pairs_kernel<false>;
        hipLaunchKernelGGL(k, grid, dim3(512), 0, s, static_cast<const float*>(wa), static_cast<const float*>(wb), D, hidden, a, b, ea, eb);
    } else {
        hipLaunchKernelGGL((mlp_weights_kernel<T>), dim3((unsigned)(((int64_t)D * hidden + 255) / 256)), dim3(256), 0, s, static_cast<const T*>(wa),
                           static_cast<const T*>(wb), D, hidden, a, b);
    }
    return launch_ok("mlp weights");
}

}  // namespace dense
}  // namespace sswin

using namespace sswin;
using namespace sswin::dense;

static int mlp_check(const char* what, int dtype, int64_t N, int D, int hidden, size_t ws_bytes, const void* ws, bool backward) {
    SSWIN_CHECK(sswin_mlp_supported(dtype, N, D, hidden), "%s: %lld rows of %d channels, %d hidden, of type %d are not supported", what, (long long)N, D, hidden,
                dtype);
    SSWIN_CHECK(ws_bytes >= sswin_mlp_workspace_bytes(dtype, D, hidden, backward) && (uintptr_t)ws % 16 == 0, "%s: the workspace is too small or not aligned", what);
    return 0;
}

// The last tile of 32 rows is moved back and read again where other wavefronts may already have stored: results lie apart from rows read
struct Rows {
    const void* p;
    size_t bytes;
};
static bool apart(std::initializer_list<Rows> results, std::initializer_list<Rows> inputs) {
    for (const Rows& r : results)
        for (const Rows& i : inputs)
            if (r.p && i.p && (uintptr_t)r.p < (uintptr_t)i.p + i.bytes && (uintptr_t)i.p < (uintptr_t)r.p + r.bytes) return false;
    return true;
}
static size_t value_size(int dtype) { return dtype == SSWIN_F32 ? 4 : 2; }

extern "C" {

int sswin_mlp_supported(int dtype, int64_t N, int D, int hidden) {
    if (N < 32 || N >= (1ll << 31) || hidden < 64 || hidden % 32 != 0) return 0;
    if (dtype == SSWIN_F32) return D == 96 && hidden <= 1024;
    if (dtype != SSWIN_F16 && dtype != SSWIN_BF16) return 0;
    return (D == 48 || D == 96) && hidden <= 1024;
}

// Where one launch is ahead of two.  16 bit: from 8192 rows on (fp16 48 channels with an fp32 residual, forward and backward: 8000 rows
// 33.4 -> 23.5 us; bf16 96 channels, 8000 rows 41.8 -> 40.0, inference 20.4 -> 18.5, 4000 rows 33.9 -> 38.4 and 16.3 -> 18.2); a wavefront's
// time grows with the hidden channels, that of the two layers' tiles with all of their work, so with more than 384 later (bf16 96 channels,
// forward and backward, 768 hidden: 20 000 rows 66 -> 76, 50 000 114 -> 91; 1024 hidden 8192 57 -> 91, 50 000 142 -> 121).  fp32: a
// wavefront takes about 44 us forward and 30 backward alone on its SIMD, so from three wavefronts a compute unit on (forward and
// backward of 8192 rows 60 -> 80 us, 16 384 88 -> 89, as three bf16 pieces; 24 576 101 -> 78, 225 700 633 -> 464), and only behind the rows up to
// which the second layer is one of few rows.
int sswin_mlp_preferred(int dtype, int64_t N, int D, int hidden) {
    if (!sswin_mlp_supported(dtype, N, D, hidden)) return 0;
    if (dtype != SSWIN_F32) return N >= (hidden <= 384 ? 8192 : 32 * hidden);
    return N > 2 * 32 * (int64_t)device_cus() && !few_rows(dtype, N, hidden, D);
}

size_t sswin_mlp_workspace_bytes(int dtype, int D, int hidden, int backward) {
    const size_t plane = (size_t)D * hidden * 2;
    return dtype == SSWIN_F32 ? 4 * plane + (size_t)(hidden + D) * sizeof(int) : backward ? 2 * plane : 0;
}

int sswin_mlp_forward(int dtype, int out_dtype, const void* x, int64_t N, int D, int hidden, const void* w1, const void* b1, const void* w2, const void* b2,
                      const void* residual, void* y, void* act, void* slope, void* ws, size_t ws_bytes, void* stream) {
    if (int rc = mlp_check("mlp_forward", dtype, N, D, hidden, ws_bytes, ws, false)) return rc;
    SSWIN_CHECK(x && w1 && w2 && y && (!act == !slope) && (ws || dtype != SSWIN_F32), "mlp_forward: null pointer");
    SSWIN_CHECK(((uintptr_t)x | (uintptr_t)w1 | (uintptr_t)b1 | (uintptr_t)w2 | (uintptr_t)b2 | (uintptr_t)residual | (uintptr_t)y | (uintptr_t)act |
                 (uintptr_t)slope) % 16 == 0, "mlp_forward: pointers must be 16-byte aligned");
    const size_t rows = (size_t)N * D * value_size(dtype), out_rows = (size_t)N * D * value_size(out_dtype), inner = (size_t)N * hidden * value_size(dtype);
    SSWIN_CHECK(apart({{y, out_rows}, {act, inner}, {slope, inner}}, {{x, rows}, {residual, out_rows}}), "mlp_forward: results may not overlap x or residual");
    hipStream_t s = static_cast<hipStream_t>(stream);
    MlpArgs g = {x, N, hidden, static_cast<const uint16_t*>(w1), static_cast<const uint16_t*>(w2), nullptr, nullptr, static_cast<const float*>(w1),
                 static_cast<const float*>(w2), b1, b2, nullptr, residual, act, slope, y, 0, 0};
    if (dtype == SSWIN_F32)
        if (int rc = launch_weights<float>(g, w1, w2, false, D, hidden, ws, s)) return rc;
#define MLP_RUN(T, TO) return act ? launch_mlp<T, TO, MLP_TRAIN>(g, D, s) : launch_mlp<T, TO, MLP_INFER>(g, D, s)
    if (dtype == SSWIN_F32 && out_dtype == SSWIN_F32) MLP_RUN(float, float);
    if (dtype == SSWIN_F16 && out_dtype == SSWIN_F16) MLP_RUN(__half, __half);
    if (dtype == SSWIN_F16 && out_dtype == SSWIN_F32) MLP_RUN(__half, float);
    if (dtype == SSWIN_BF16 && out_dtype == SSWIN_BF16) MLP_RUN(__hip_bfloat16, __hip_bfloat16);
    if (dtype == SSWIN_BF16 && out_dtype == SSWIN_F32) MLP_RUN(__hip_bfloat16, float);
#undef MLP_RUN
    return fail("mlp_forward: operands of type %d with a result of type %d are not supported", dtype, out_dtype);
}

int sswin_mlp_backward(int dtype, const void* dy, int64_t N, int D, int hidden, const void* w1, const void* w2, const void* slope, void* du, void* dx, void* ws,
                       size_t ws_bytes, void* stream) {
    if (int rc = mlp_check("mlp_backward", dtype, N, D, hidden, ws_bytes, ws, true)) return rc;
    SSWIN_CHECK(dy && w1 && w2 && slope && du && dx && ws, "mlp_backward: null pointer");
    SSWIN_CHECK(((uintptr_t)dy | (uintptr_t)w1 | (uintptr_t)w2 | (uintptr_t)slope | (uintptr_t)du | (uintptr_t)dx) % 16 == 0,
                "mlp_backward: pointers must be 16-byte aligned");
    const size_t rows = (size_t)N * D * value_size(dtype), inner = (size_t)N * hidden * value_size(dtype);
    SSWIN_CHECK(apart({{du, inner}, {dx, rows}}, {{dy, rows}, {slope, inner}}), "mlp_backward: results may not overlap dy or slope");
    hipStream_t s = static_cast<hipStream_t>(stream);
    MlpArgs g = {dy, N, hidden, nullptr, nullptr, nullptr, nullptr, static_cast<const float*>(w2), static_cast<const float*>(w1), nullptr, nullptr, slope,
                 nullptr, du, nullptr, dx, 0, 0};
#define MLP_RUN(T)                                                                      \
    do {                                                                                \
        if (int rc = launch_weights<T>(g, w2, w1, true, D, hidden, ws, s)) return rc;   \
        return launch_mlp<T, T, MLP_BACKWARD>(g, D, s);                                 \
    } while (0)
    if (dtype == SSWIN_F32) MLP_RUN(float);
    if (dtype == SSWIN_F16) MLP_RUN(__half);
    MLP_RUN(__hip_bfloat16);
#undef MLP_RUN
}

}  // extern "C"
