// What flash_window.hip, the attention kernels that take a window and head a wavefront, is made of: the pieces of work of a workgroup, LDS and rows, D = dO . O,
// pairs of fp16 and their scales, the units of the bias table's sums.
#pragma once

#include <math.h>

#include <algorithm>
#include <type_traits>

#include "flash_common.hpp"

namespace sswin {
namespace flash {
namespace window {

constexpr int HD = 16, WAVES = 4, MOST = 24;                             // channels of a head; wavefronts of a workgroup; tiles of 16 tokens of a window
constexpr int DELTA_BLOCKS = 1024, FORWARD_BLOCKS = 1024;
constexpr int MOST_HEADS = FORWARD_BLOCKS / 8;                           // workgroups of a head come in eights
constexpr int LIST_HEAD = 32, LIST_THREADS = 1024, LIST_WINDOWS = 16384;
constexpr uint32_t INDEX = 0x7ffcu;                                      // of a difference of words: 4 row of the table
constexpr int PITCH = 20, TURN = 16 * PITCH;                             // a 16 x 16 tile in LDS, values
static_assert(MAX_ROWS * 4 <= 1 << 15, "codes and regions share a word");
static_assert(MOST <= LIST_HEAD - 2, "the list's head counts windows by their tiles");

struct Args {
    const int32_t* plan;       // group table: [c | T | ..] of g_cap entries each, window k's groups at k H
    int64_t g_cap;
    const int32_t* order;      // voxel of token rank r
    const uint32_t* word;      // 4 code | region << 15 | several regions in the window << 31 of token r
    const int32_t* list;       // [t]: windows of more than t tiles; from LIST_HEAD on the windows, largest first
    float* largest_v;          // largest |V| of the forward's workgroups, n_largest_v a head
    int n_largest_v;
    int64_t N;
    int windows, H, rows, offset4, per_head;
    float scale;
    const float* table;        // [rows, H]
    const void* qkv;           // [N, 3 H hd] voxel rows
    void* out;                 // [N, H hd]
    float* lse;                // [H, N] by rank: offset + log2 of the row sum
    // backward
    const void* dout;          // [N, H hd]
    const float* delta;        // [N, H]: dO . O
    void* dqkv;                // [N, 3 H hd]
    const float* largest;      // [H, n_largest] largest |dO| of a head in some tokens
    int n_largest;
    int bits;                  // a sum of the bias table's gradient takes values below 2^bits units
    float* partial;            // [H][per_head][rows] sums of dS by table row
};

// Workgroup -> head and place among the head's workgroups: the heads of the same windows follow each other on one XCD, whose L2 holds their rows
__device__ __forceinline__ void place(int H, int& h, int& first) {
    const int b = (int)blockIdx.x, y = b >> 3;
    h = y % H;
    first = y / H * 8 + (b & 7);
}

// The head's column of the bias table in units of log 2
__device__ __forceinline__ void stage_table(const Args& g, int h, float* bias) {
    constexpr int AT_ONCE = 9;                                           // of a thread, requested together: 13^3 rows
    for (int r0 = threadIdx.x; r0 < g.rows; r0 += WAVES * 64 * AT_ONCE) {
        float v[AT_ONCE];
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i) v[i] = g.table[(int64_t)min(r0 + i * WAVES * 64, g.rows - 1) * g.H + h];
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i)
            if (r0 + i * WAVES * 64 < g.rows) bias[r0 + i * WAVES * 64] = v[i] * LOG2E;
    }
}

// The pieces of work of a workgroup, as its wavefronts have them: every per_head-th of its head.  The largest windows come first, a workgroup
// each; then those that two wavefronts hold, two at a time; then four at a time.  Lane l holds what is known of the l-th piece: list and plan are read
// once, in front of the work.
struct Task {
    int team, rank, steps;     // wavefronts on the window, this one's number, tiles of the largest window among the workgroup's
    int c, T, first, tiles;    // the window's tokens (0: nothing to do) and first rank, this wavefront's tiles
};
// TILES: of one wavefront; a window of up to 2 TILES has two, a larger one all four
template <int TILES> struct Work {
    int r0, left, at;          // first round in the lanes, rounds in them, lane of the next one
    int own, team, steps, c, T;
    // Rounds of pieces by descending size, every other one from behind: first come, first served would give the first workgroups the larger of every round
    // (windows of 7^3: the longest wavefront of the backward 1.44 times the mean with 112 700 voxels fp32, 116 -> 102 us; 225 700 fp16 149 -> 143)
    __device__ __forceinline__ void load(const Args& g) {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = r0 + lane, u = r * g.per_head + (r & 1 ? g.per_head - 1 - own : own);
        const int big = g.list[2 * TILES], two = g.list[TILES], pairs = (two - big + 1) / 2, total = big + pairs + (g.windows - two + WAVES - 1) / WAVES;
        left = __builtin_popcountll(__ballot(u < total));
        at = team = steps = c = T = 0;
        if (u >= total) return;
        int from, end;
        if (u < big) team = 4, from = u, end = big;
        else if (u < big + pairs) team = 2, from = big + 2 * (u - big), end = two;
        else team = 1, from = two + WAVES * (u - big - pairs), end = g.windows;
        const int window = from + wave / team;
        const int64_t head = (int64_t)g.list[LIST_HEAD + from] * g.H, group = (int64_t)g.list[LIST_HEAD + min(window, g.windows - 1)] * g.H;
        steps = (g.plan[head] + 15) >> 4;
        c = window < end ? g.plan[group] : 0;
        T = g.plan[g.g_cap + group];
    }
    __device__ __forceinline__ Work(const Args& g, int first) {
        own = first, r0 = 0;
        load(g);
    }
    __device__ __forceinline__ bool next(const Args& g, Task& t) {
        if (at == 64) {
            r0 += 64;
            load(g);
        }
        if (at >= left) return false;
        t.team = __builtin_amdgcn_readlane(team, at);
        t.steps = __builtin_amdgcn_readlane(steps, at);
        t.c = __builtin_amdgcn_readlane(c, at);
        t.T = __builtin_amdgcn_readlane(T, at);
        ++at;
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), all = (t.c + 15) >> 4, shift = t.team >> 1, share = all >> shift,
                  more = all - (share << shift);
        t.rank = wave & (t.team - 1);
        t.tiles = share + (t.rank < more ? 1 : 0);
        t.first = t.rank * share + min(t.rank, more);
        return true;
    }
};

__device__ __forceinline__ f32x4 widened(const Frag<float>& f) { return f.v; }
__device__ __forceinline__ f32x4 widened(const Frag<__half>& f) { return f32x4{(float)f.v[0], (float)f.v[1], (float)f.v[2], (float)f.v[3]}; }
__device__ __forceinline__ f32x4 widened(const Frag<__hip_bfloat16>& f) {
    const uint2 w = __builtin_bit_cast(uint2, f.v);
    return f32x4{__builtin_bit_cast(float, w.x << 16), __builtin_bit_cast(float, w.x & 0xffff0000u), __builtin_bit_cast(float, w.y << 16),
                 __builtin_bit_cast(float, w.y & 0xffff0000u)};
}

// Between a store to LDS of the wavefront's own and what other lanes read there, and the other way round: no instruction, but the compiler, which sees a
// lane's own addresses alone, exchanges nothing across it
__device__ __forceinline__ void lanes_meet() { __builtin_amdgcn_wave_barrier(); }
// a 16 x 16 tile turned through LDS of the wavefront's own: lane (row l % 16, columns 4 (l / 16) + j) -> lane (rows 4 (l / 16) + j, column l % 16)
__device__ __forceinline__ f32x4 turned(float* tile, const f32x4& v) {
    const int l16 = threadIdx.x & 15, quad = (threadIdx.x & 63) >> 4;
    *reinterpret_cast<f32x4*>(tile + l16 * PITCH + quad * 4) = v;
    lanes_meet();
    f32x4 r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = tile[(quad * 4 + j) * PITCH + l16];
    lanes_meet();
    return r;
}

// over the four lanes l % 16, to all of them
template <typename F> __device__ __forceinline__ float across(float v, F&& f) {
    const auto a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    v = f(__builtin_bit_cast(float, (uint32_t)a[0]), __builtin_bit_cast(float, (uint32_t)a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    return f(__builtin_bit_cast(float, (uint32_t)b[0]), __builtin_bit_cast(float, (uint32_t)b[1]));
}
__device__ __forceinline__ float across_max(float v) {
    return across(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float across_sum(float v) {
    return across(v, [](float a, float b) { return a + b; });
}

// LDS by its address: a word of a query less one of a key is the address of their bias
typedef __attribute__((address_space(3))) float LdsFloat;
typedef __attribute__((address_space(3))) unsigned long long LdsLong;
__device__ __forceinline__ uint32_t lds_address(const void* p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p; }
__device__ __forceinline__ float lds_float(uint32_t at) { return *(const LdsFloat*)(uintptr_t)at; }

// Arrays through buffer descriptors: a lane's 32 bits of offset and one of all lanes, no 64-bit addresses in vector registers, and what is read behind
// an array's end is 0 (the clamps of the last step's rows).
typedef __amdgpu_buffer_rsrc_t Buffer;
template <typename V> __device__ __forceinline__ Buffer buffer(const V* p, int64_t count) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<V*>(p), 0, (int)(uint32_t)(count * (int64_t)sizeof(V)), 0x00020000);
}
__device__ __forceinline__ uint32_t load1(const Buffer& b, uint32_t lane_bytes, uint32_t bytes) {
    return __builtin_amdgcn_raw_buffer_load_b32(b, lane_bytes, bytes, 0);
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u32x4 load4(const Buffer& b, uint32_t lane_bytes, uint32_t bytes) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(b, lane_bytes, bytes, 0));
}
// rows of the voxels' tokens: four of a head's channels a lane
template <typename T> struct Rows {
    Buffer b;
    uint32_t pitch, col, own;  // bytes: a row, the head's first channel, the lane's first channel in it
    __device__ __forceinline__ Rows(const void* p, int64_t N, int pitch_, int col_)
        : b(buffer(static_cast<const T*>(p), N * pitch_)), pitch((uint32_t)pitch_ * (uint32_t)sizeof(T)), col((uint32_t)col_ * (uint32_t)sizeof(T)),
          own(((threadIdx.x & 63) >> 4) * (uint32_t)(4 * sizeof(T))) {}
    __device__ __forceinline__ void row(int v, Frag<T>& f) const {
        const uint32_t at = __umul24((uint32_t)v, pitch) + own;
        if constexpr (sizeof(T) == 4) f.v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(b, at, col, 0));
        else f.v = __builtin_bit_cast(decltype(f.v), __builtin_amdgcn_raw_buffer_load_b64(b, at, col, 0));
    }
    // The whole offset in the lane's register.  With a part of it in a scalar one the compiler puts no wait between a store of 16 bytes and an instruction that
    // writes the registers it stores, and the new value is what arrives (heads of 32 once stored so: 1 value of 1000 was that of the next 16 channels).
    __device__ __forceinline__ void store(int v, const f32x4& x) const {
        const uint32_t at = __umul24((uint32_t)v, pitch) + (own + col);
        if constexpr (sizeof(T) == 4) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), b, at, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, packed<T>(x).v), b, at, 0, 0);
    }
};
template <typename T> __device__ __forceinline__ void keep(bool live, Frag<T>& f) {
    if (!live) f = Frag<T>{};
}
// the largest |x| of a row's four values, 0 if one of them is infinite
__device__ __forceinline__ float largest_finite(const f32x4& v) {
    const float m = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
    return m < INFINITY ? m : 0.f;
}
__device__ __forceinline__ float largest_of_workgroup(float m, float* part) {
    for (int o = 1; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    m = part[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) m = fmaxf(m, part[w]);
    return m;
}
// 0, or NaN if one of them is not finite
__device__ __forceinline__ float not_finite(const f32x4& v) { return fmaf(v[0], 0.f, fmaf(v[1], 0.f, fmaf(v[2], 0.f, v[3] * 0.f))); }

// ------------------------------------------------------------------------------------------
// D = dO . O of every voxel and head, HD / 4 lanes a head, and the largest |dO| (of what is finite) of a workgroup and head.  A lane keeps to one head: lanes
// behind the last whole number of voxels that the launch holds have nothing to do.
// ------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void flash_window_delta_kernel(const T* __restrict__ dout, const T* __restrict__ out, int64_t parts, int H, float* __restrict__ delta,
                                                                 float* __restrict__ largest) {
    __shared__ uint32_t of_head[MOST_HEADS];
    constexpr int AT_ONCE = 4, LANES = HD / 4;
    for (int i = threadIdx.x; i < H; i += 256) of_head[i] = 0;
    const int row = (int)(blockIdx.x * 256 + threadIdx.x) / LANES, stride = (int)(gridDim.x * (256 / LANES)) / H * H * LANES;
    float most = 0.f;
    if (row * LANES < stride) {
        for (int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x; i0 < parts; i0 += (int64_t)stride * AT_ONCE) {
            Frag<T> x[AT_ONCE], y[AT_ONCE];
#pragma unroll
            for (int k = 0; k < AT_ONCE; ++k) {
                const int64_t i = i0 + (int64_t)stride * k, j = i < parts ? i : i0;   // (of the lane's head too)
                x[k].load(dout + j * 4), y[k].load(out + j * 4);
            }
#pragma unroll
            for (int k = 0; k < AT_ONCE; ++k) {
                const int64_t i = i0 + (int64_t)stride * k;
                const f32x4 a = widened(x[k]), b = widened(y[k]);
                float dot = 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j) dot = fmaf(a[j], b[j], dot);
                dot += dpp_f32<0xB1>(dot);
                dot += dpp_f32<0x4E>(dot);
                most = fmaxf(most, largest_finite(a));
                if (i < parts && (threadIdx.x & (LANES - 1)) == 0) delta[i / LANES] = dot;
            }
        }
    }
    __syncthreads();
    if (most > 0.f) atomicMax(&of_head[row % H], __builtin_bit_cast(uint32_t, most));   // (bits grow with the value)
    __syncthreads();
    for (int i = threadIdx.x; i < H; i += 256) largest[(int64_t)i * gridDim.x + blockIdx.x] = __builtin_bit_cast(float, of_head[i]);
}

// The units of the table's sums.  Integers, so that the result does not depend on the order of the additions.  A head's |dS| <= |dP| + |D| <= 2 HD largest |dO|
// largest |V| (P of a row adds up to at most one, up to rounding) < 2^top, whole numbers below 2^bits in units of 2^(top - bits); a workgroup adds at most
// 2^(62 - bits) of them to a row of the table.  A value below 2^KEEPS units would lose bits of its fp32 there: it is added to a second sum, in units
// 2^(bits - KEEPS) as fine.  So every value down to 2^(2 KEEPS - 2 bits) of the bound is added as exactly as fp32 has it, wherever the head's largest dO and V lie.
// (One sum in units of all heads' largest: a row of dO in one head and one of V in another, 2^20 above the rest, left nothing of the others' dS.)  What the second
// sum costs the backward, three instructions a value, windows of 7^3: 112 700 tokens fp32 115 -> 117 us, fp16 88 -> 91, 8100 in nearly full windows fp32 154 -> 163.
constexpr int KEEPS = 23;
__device__ __forceinline__ int bound_of_ds(float mo, float mv) {
    return (mo > 0.f ? (int)ilogbf(mo) : -149) + (mv > 0.f ? (int)ilogbf(mv) : -149) + 8;
}

// ------------------------------------------------------------------------------------------
// Pieces.  P, dS and, of fp32 tokens, the rows are multiplied on the 16-bit matrix cores as pairs of fp16 rounded to nearest, products of two second pieces left
// out of dQ alone; sums are fp32.  Rows are x 2^e = h + l, 22 bits or 2^-25 in their scale, whichever is more.  A scale e is one of a wavefront: of K and V for
// the window, of Q and dO kept from step to step until a row no longer fits, when the sums so far are scaled with it.  Rows too far below the largest for
// that, and windows in which something is not finite, are done with fp32 products (How::exact), a whole window at a time.  Where that is nearly every window, backward with
// the table's gradient, 114 000 tokens in windows of 7^3: 1 % of the rows of dO or of K 2^-14 of the others, fp32 125 -> 214 us (chunks of 32 tokens: 237); rows of dO
// spread by e^(3 randn), fp32 125 -> 209, fp16 101 -> 165 (169).
// P and dS have no scale of their own, and a row of dS is as much smaller than another as its row of dO, or as its P: x = h + l 2^-11, 22 bits down to 2^-14
// and 2^-36 below that (with the pieces of a row for them, 22 bits or 2^-25 in a window's scale, dQ of a query whose dO is 2^-9 of the window's largest was off
// by 1.6e-5).  Error of a row against float64, its norm, median, windows of 7^3, fp32: dQ 6.4e-7 with fp32 products, 2.8e-7 here, dK 6.3 and 3.4, dV 6.2 and 3.3, the same
// for rows of dO 2^-9 of the others and for mask regions that hold nothing else; the table's gradient, by head, 5.7 and 3.0.  16-bit tokens: the rounding of the result.
// ------------------------------------------------------------------------------------------
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
struct Pair {                  // x = h + l
    f16x4 h, l;
};
__device__ __forceinline__ Pair split(const f32x4& x) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    struct Words { uint32_t a, b; };
    Words h, l;
    f16x2 h0 = {(_Float16)x[0], (_Float16)x[1]}, h1 = {(_Float16)x[2], (_Float16)x[3]};
    asm("" : "+v"(h0), "+v"(h1));                                        // (or each half is converted again for its rest)
    const f16x2 l0 = {(_Float16)fmaf(-1.f, (float)h0[0], x[0]), (_Float16)fmaf(-1.f, (float)h0[1], x[1])};
    const f16x2 l1 = {(_Float16)fmaf(-1.f, (float)h1[0], x[2]), (_Float16)fmaf(-1.f, (float)h1[1], x[3])};
    h = {__builtin_bit_cast(uint32_t, h0), __builtin_bit_cast(uint32_t, h1)};
    l = {__builtin_bit_cast(uint32_t, l0), __builtin_bit_cast(uint32_t, l1)};
    return Pair{__builtin_bit_cast(f16x4, h), __builtin_bit_cast(f16x4, l)};
}
struct Fine {                  // x = h + l / REST
    f16x4 h, l;
};
constexpr float REST = 2048.f;
// of x 2^MORE
template <int MORE = 0> __device__ __forceinline__ Fine split_fine(const f32x4& x) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    struct Words { uint32_t a, b; };
    constexpr float BY = (float)(1 << MORE);
    Words h, l;
    f16x2 h0 = {(_Float16)(x[0] * BY), (_Float16)(x[1] * BY)}, h1 = {(_Float16)(x[2] * BY), (_Float16)(x[3] * BY)};
    asm("" : "+v"(h0), "+v"(h1));                                        // (as above)
    const f16x2 l0 = {(_Float16)fmaf(-REST, (float)h0[0], x[0] * (BY * REST)), (_Float16)fmaf(-REST, (float)h0[1], x[1] * (BY * REST))};
    const f16x2 l1 = {(_Float16)fmaf(-REST, (float)h1[0], x[2] * (BY * REST)), (_Float16)fmaf(-REST, (float)h1[1], x[3] * (BY * REST))};
    h = {__builtin_bit_cast(uint32_t, h0), __builtin_bit_cast(uint32_t, h1)};
    l = {__builtin_bit_cast(uint32_t, l0), __builtin_bit_cast(uint32_t, l1)};
    return Fine{__builtin_bit_cast(f16x4, h), __builtin_bit_cast(f16x4, l)};
}
__device__ __forceinline__ f16x8 both(const f16x4& a, const f16x4& b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }
// x and x / REST: one product with both pieces of a Fine adds them in their scales
__device__ __forceinline__ f16x8 with_rest(const f16x4& x) { return both(x, x * (_Float16)(1.f / REST)); }
__device__ __forceinline__ f16x8 both(const Fine& x) { return both(x.h, x.l); }
__device__ __forceinline__ f16x4 halves(const f32x4& x) { return packed<__half>(x).v; }
__device__ __forceinline__ f32x4 mma32(const f16x8& a, const f16x8& b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x4 mma16(const f16x4& a, const f16x4& b, const f32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0); }

// Powers of two that bring numbers into fp16's range: `e` for a largest value of [2^(12 - e), 2^(13 - e)), kept until it reaches 2^(15 - e)
constexpr uint32_t NOT_FINITE = 0x7f800000u;
__device__ __forceinline__ float power(int e) { return __builtin_bit_cast(float, (uint32_t)(127 + e) << 23); }
__device__ __forceinline__ uint32_t largest4(const f32x4& v) {           // as bits, which grow with the absolute value
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float x = v[j];                                            // (a bit cast of the element itself takes the first)
        m = max(m, __builtin_bit_cast(uint32_t, x) & 0x7fffffffu);
    }
    return m;
}
__device__ __forceinline__ uint32_t over_quads(uint32_t m) {             // the largest of the four lanes l % 16
    const auto a = __builtin_amdgcn_permlane16_swap(m, m, false, false);
    m = max((uint32_t)a[0], (uint32_t)a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(m, m, false, false);
    return max((uint32_t)b[0], (uint32_t)b[1]);
}
__device__ __forceinline__ int over_rows(uint32_t m) {                   // of all lanes, once over_quads has been
    m = m < NOT_FINITE ? m : 0;
    return __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, row16_max(__builtin_bit_cast(float, m))));
}
__device__ __forceinline__ int scale_for(int largest, int most) { return largest == 0 ? most : max(-most, min(most, 12 + 127 - (largest >> 23))); }
__device__ __forceinline__ bool too_large(uint32_t m, int e) { return m >= (uint32_t)(142 - e) << 23; }
// pieces of a row whose largest value is below 2^(low - e) would lose bits of it: fp32 rows any below 22; 16-bit rows, of 8 or 11 bits in one piece that keeps 2^-25, those
// below 2^-10, where P dO and dS, the second piece in 2^-36, still have some 15.  (2^-6 until dS had its finer pieces.)
template <typename T> __device__ __forceinline__ bool too_small(uint32_t m, int e) {
    constexpr int low = sizeof(T) == 4 ? 0 : -10;
    return m != 0 && m < (uint32_t)(127 + low - e) << 23;
}

// Workgroups of a head: as many as find a place at once, and no more than it has windows
inline int per_head(int windows, int H, int resident) {
    const int m = std::max(1, resident * device_cus() / (8 * H));
    return std::min(8 * m, (windows + 7) / 8 * 8);
}

}  // namespace window
}  // namespace flash
}  // namespace sswin
