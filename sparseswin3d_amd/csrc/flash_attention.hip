// Window attention for windows of any size with heads of 16 or 32 channels, the attention matrix kept in registers
// (WindowAttention.forward, sparse_swin/swin3d_base.py:654-675, from the projected qkv to the attention output, and its
// backward).  It serves what the kernels of window_attention.hip do not take: heads of 16 channels, windows of more than 128
// positions (the reference's own setting: 7^3 windows, heads of 16).
// Heads of 16 in windows of up to 384 positions run on flash_window.hip.
//
// Work: the token ranks (sorted by window) are cut into chunks of 32 and a wavefront owns the blocks that start in its chunk:
// 32 tokens of a large window, or several small windows together up to 32 tokens, so that sparse scenes do not pay a tile
// per window.  A block walks over the tokens of its window(s) 16 at a time; all products are 16 x 16 tiles, so that padding
// stops at 16 rows.  No task list, no barrier in the loop; the next 16 rows are covered by the other wavefronts of the SIMD.
//
// Layouts: v_mfma_f32_16x16x*: operand lane l = (row l % 16, reduction slots 4 (l / 16) + j), accumulator lane l = (column
// l % 16, rows 4 (l / 16) + r).  An accumulator packed in place is therefore the operand of the next product over its rows:
// S^T = K Q^T gives P^T as the operand of O^T = V^T P^T, and the row of a query (its maximum, sum and rescaling) lies in the
// four lanes l % 16.  fp32 tokens take four 16x16x4 fp32 products per 16 slots, products of two 16-bit tokens one 16x16x16.  P
// and dS stay fp32 for 16-bit tokens as well (as in the operators; dS of fp16 tokens would leave fp16's range): their products
// are the fp32 ones, with the tokens widened.
//
// Softmax as the operators define it: exp(s - m) / (sum exp(s - m) + 1e-8), m = max(0, row maximum).  The running offset is the
// maximum over the first 16 tokens (exponentials of its rows are of order one, however far below 0 the scores lie) and moves only when
// a score exceeds it by 10 in units of log 2: a row usually needs one exchange between its lanes at the start and one at the
// end, where the 1e-8 is scaled to the offset that was used.
//
// The relative position bias is read from the table of the head in LDS: index of (p, q) = code[p] - code[q] + offset.  A token
// carries {4 code, mask region, window} in one word, so one subtraction gives the table address and whether mask or window
// differ.
//
// Backward: with dS asked for (the bias table's gradient needs it) the key side forms scores, P and dS, sums dV and dK and stores
// dS, and the query side is dQ = dS K from the stored dS; before, both sides formed them and the query side stored.
//
// 112 700 voxels, windows of 7^3, 3 heads of 16 (27 million scores): fp32 forward 56 us, backward 172 (D 11, key side 117,
// dQ 43; 63 and 178 with the work taken by rank).  225 700 voxels, fp16: forward 80 us, backward 285 (14, 180, 91; dS is 217 MB written and read again).  dQ waits for
// memory, 15 us a wavefront of four 32 x 32 pieces; rows of dS padded to 64 bytes, rows read by neighbouring
// lanes and exchanged, voxels kept in lanes change it by less than 3 %.  The block products with the attention matrix in memory take 195 and 258 us (112 700 voxels, fp32).  The vector ALU is
// busy for half of a launch, the fp32 matrix instructions (which occupy it) for another quarter; leaving out the bias reads, the
// exponentials or the row loads one by one changes the forward by less than 3 %, the rows of the backward by 15 %.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "flash_common.hpp"

namespace sswin {
namespace flash {

constexpr int WAVES = 4;
constexpr int TOKENS_WAVES = 16, ORDER_THREADS = TOKENS_WAVES * 64, ORDER_CLASSES = 16, ORDER_MOST = 12288, ORDER_WINDOWS = 16384;

struct Args {
    const int32_t* order;      // voxel of token rank r
    const int32_t* tok_T;      // rank of the first token of r's window
    const int32_t* tok_c;      // tokens of r's window
    const uint32_t* word;      // 4 code | region << 15 | first rank << 23 | several regions << 31 of token r (flash_tokens_kernel)
    int64_t N;
    int H, rows, offset4;
    float scale;               // of the scores
    const float* table;        // [rows, H]
    const void* qkv;           // [N, 3 H hd] voxel rows
    void* out;                 // [N, H hd]
    float* lse;                // [H, N] by rank: offset + log2 of the row sum
    // backward
    const void* dout;          // [N, H hd]
    float* delta;              // [H, N] by rank: dO . O
    void* dqkv;                // [N, 3 H hd]
    float* ds;                 // [c x c] blocks of the groups, or null
    const int32_t* tok_sq;     // sum of c * c over the windows before r's
    const int32_t* work;       // chunks in the order they are taken, or null: by their ranks
};

// The chunks by descending work, those of equal work by their ranks (a window's stay together), by one workgroup.  A chunk's work follows from its window's
// size, 1 to 22 steps, and the four wavefronts of a workgroup hold their place until the last is done: taken by their ranks, 61 to 69 %
// of the places are in use, by descending work 89 to 97 % (simulated on the rooms of 112 700 and 225 700 voxels; 69 % measured).
// 112 700 voxels fp32: forward 62.8 -> 56.0 us, key side 126.9 -> 117.3, dQ 42.9 either way (by rank behind an ordered key side 45.9); 225 700 fp16: forward
// 89.4 -> 79.5, key side 182 -> 180.  The launch for the words takes 6.4 and 9.1 us with the order, 4.2 and 4.4 without (alone; inside a module 7.4 and 10).
// The work is summed over the windows (their table is short; 7055 chunks of the token rows take one workgroup 40 us): a step of 16 tokens of the window counts
// two, three with a second sub-tile, a block two more; windows of less than 32 tokens, which share blocks, count by their tokens.
__device__ __forceinline__ void order_chunks(const int32_t* __restrict__ plan, int64_t g_cap, int64_t windows, int H, int64_t N, int32_t* __restrict__ work) {
    __shared__ uint32_t cost[ORDER_MOST / 2];                            // two chunks each
    __shared__ uint16_t place[ORDER_CLASSES * ORDER_THREADS];            // [class][thread]
    __shared__ int sums[TOKENS_WAVES];
    const int chunks = (int)((N + 31) / 32), t = threadIdx.x;
    if (windows > ORDER_WINDOWS) {
        for (int i = t; i < chunks; i += ORDER_THREADS) work[i] = i;
        return;
    }
    for (int i = t; i < (chunks + 1) / 2; i += ORDER_THREADS) cost[i] = 0;
    __syncthreads();
    auto add = [&](int rank, int v) { atomicAdd(&cost[rank >> 6], (uint32_t)v << (rank >> 1 & 16)); };
    for (int k = t; k < (int)windows; k += ORDER_THREADS) {
        const int c = plan[(int64_t)k * H], T = plan[g_cap + (int64_t)k * H];
        if (c < 32) add(T, (c + 7) / 8);
        else
            for (int j = 0; j < c; j += 32) add(T + j, (c + 15) / 16 * (c - j > 16 ? 3 : 2) + 2);
    }
    __syncthreads();
    auto kind = [&](int i) { return ORDER_CLASSES - 1 - min((int)(cost[i >> 1] >> ((i & 1) * 16) & 0xffffu) / 4, ORDER_CLASSES - 1); };
    for (int k = 0; k < ORDER_CLASSES; ++k) place[k * ORDER_THREADS + t] = 0;
    __syncthreads();
    const int per = (chunks + ORDER_THREADS - 1) / ORDER_THREADS, begin = min(t * per, chunks), end = min(begin + per, chunks);
    for (int i = begin; i < end; ++i) ++place[kind(i) * ORDER_THREADS + t];
    __syncthreads();
    // sums in front, classes first; a thread adds 16 neighbours
    int own = 0;
    for (int k = 0; k < ORDER_CLASSES; ++k) own += place[t * ORDER_CLASSES + k];
    int before = own;
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(before, o, 64);
        if ((t & 63) >= o) before += v;
    }
    if ((t & 63) == 63) sums[t >> 6] = before;
    __syncthreads();
    before -= own;
    for (int w = 0; w < t >> 6; ++w) before += sums[w];
    for (int k = 0; k < ORDER_CLASSES; ++k) {
        const int n = place[t * ORDER_CLASSES + k];
        place[t * ORDER_CLASSES + k] = (uint16_t)before;
        before += n;
    }
    __syncthreads();
    for (int i = begin; i < end; ++i) work[place[kind(i) * ORDER_THREADS + t]++] = i;
}

// What a token contributes to the table index, mask and window comparisons, one word per rank, and the sum of c * c over
// the windows before its own; a wavefront per window.  The first workgroup finds the chunks' order, if it is asked for.
__global__ __launch_bounds__(ORDER_THREADS) void flash_tokens_kernel(const int32_t* __restrict__ plan, int64_t g_cap, int64_t windows, int H,
                                                                     const int32_t* __restrict__ tok_pos, int64_t N, const int32_t* __restrict__ code,
                                                                     const int8_t* __restrict__ mask, int nmw, int n, uint32_t* __restrict__ word,
                                                                     int32_t* __restrict__ tok_sq, int32_t* __restrict__ work) {
    int64_t block = blockIdx.x;
    if (work && block-- == 0) return order_chunks(plan, g_cap, windows, H, N, work);
    const int64_t k = block * TOKENS_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (k >= windows) return;
    const int64_t g = k * H;                                             // the window's first group (head 0)
    const int c = plan[g], T = plan[g_cap + g], sq = plan[2 * g_cap + g] / H, w = plan[3 * g_cap + g];
    const int8_t* region = mask ? mask + (int64_t)(w % nmw) * n : nullptr;
    uint32_t several = 0;                                                // several regions in this window
    if (region) {
        const int8_t r0 = region[tok_pos[T]];
        bool differ = false;
        for (int i = threadIdx.x & 63; i < c; i += 64) differ = differ || region[tok_pos[T + i]] != r0;
        several = __any(differ) ? 0x80000000u : 0u;
    }
    for (int i = threadIdx.x & 63; i < c; i += 64) {
        const int p = tok_pos[T + i];
        word[T + i] = (uint32_t)code[p] * 4u | (region ? ((uint32_t)(uint8_t)region[p]) << 15 : 0u) | ((uint32_t)T & 0xffu) << 23 | several;
        if (tok_sq) tok_sq[T + i] = sq;
    }
}

// Block of work: own ranks [a, a + len), the ranks [from, to) of the windows they belong to
struct Block {
    int a, len, from, to;
    bool merged;               // several windows
};

// The blocks that start in the 32 ranks of a chunk, one after the other.  Lane l holds what is known of rank r0 + l (a block
// may reach 31 ranks past its chunk); all of it is requested together, before the bias table is waited for.
//
// Values that are not finite: 0 x inf is NaN, so one of them in a row that takes part with P = 0 (another window of a merged block,
// the repeated rows behind a window's end) or in a product with the identity would spread.  The kernels look at a block's results:
// where one is NaN the block is done again, and the rest of the chunk after it, one window at a time with columns read lane by
// lane and nothing behind the end.  Finite tokens pay one comparison a block.
struct Blocks {
    int r0, T, c, voxel;
    uint32_t word, starts, before;
    bool careful;
    __device__ __forceinline__ Blocks(const Args& g, int64_t chunk) {
        r0 = (int)(chunk * 32);
        const int r = r0 + (int)(threadIdx.x & 63), at = (int)(r < g.N ? r : g.N - 1);
        T = g.tok_T[at];
        c = g.tok_c[at];
        voxel = g.order[at];
        word = g.word[at];
    }
    __device__ __forceinline__ void begin(const Args& g) {
        const int lane = threadIdx.x & 63, r = r0 + lane;
        starts = (uint32_t)__ballot(lane < 32 && r < g.N && ((r - T) & 31) == 0);
        careful = false;
    }
    // the block next() returned last once more, if a sum of its results is NaN
    __device__ __forceinline__ bool again(float sum) {
        if (careful || !__any(sum != sum)) return false;
        starts = before;
        return careful = true;
    }
    // of the block's own token s * 16 + l % 16 (the last one again behind it)
    __device__ __forceinline__ int slot(const Block& b, int s) const { return b.a - r0 + min(s * 16 + (int)(threadIdx.x & 15), b.len - 1); }
    __device__ __forceinline__ bool next(Block& b) {
        if (!starts) return false;
        before = starts;
        int j = __builtin_ctz(starts);
        starts &= starts - 1;
        const int T0 = __builtin_amdgcn_readlane(T, j), c0 = __builtin_amdgcn_readlane(c, j);
        b.a = r0 + j;
        b.from = T0;
        b.to = T0 + c0;
        b.merged = false;
        if (c0 >= 32) {
            b.len = min(32, b.to - b.a);
            return true;
        }
        // small windows that follow each other share a block as long as they fit
        while (starts && !careful) {
            j = __builtin_ctz(starts);
            const int cn = __builtin_amdgcn_readlane(c, j);
            if (cn >= 32 || b.to - b.a + cn > 32) break;
            starts &= starts - 1;
            b.to += cn;
            b.merged = true;
        }
        b.len = b.to - b.a;
        return true;
    }
};

__device__ __forceinline__ float across(float v, bool maximum) {         // over the four lanes that hold a column
    float o = __shfl_xor(v, 16, 64);
    v = maximum ? fmaxf(v, o) : v + o;
    o = __shfl_xor(v, 32, 64);
    return maximum ? fmaxf(v, o) : v + o;
}

template <int NB> __device__ __forceinline__ float sum_of(const f32x4 (&o)[2][NB]) {
    float t = 0.f;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int c = 0; c < NB; ++c) t += (o[s][c][0] + o[s][c][1]) + (o[s][c][2] + o[s][c][3]);
    return t;
}

// Workgroup -> head and first chunk: the heads of the same tokens follow each other on one XCD, whose L2 holds their rows
__device__ __forceinline__ void place(int H, int64_t groups, int& h, int64_t& first) {
    const int64_t b = blockIdx.x, full = groups / 8 * 8 * H;
    if (b < full) {
        const int64_t i = b / 8;
        h = (int)(i % H);
        first = (i / H * 8 + b % 8) * WAVES;
    } else {
        const int64_t i = b - full, rest = groups % 8;
        h = (int)(i / rest);
        first = (groups / 8 * 8 + i % rest) * WAVES;
    }
}

__device__ __forceinline__ int64_t chunk_of(const Args& g, int64_t at) { return g.work && at * 32 < g.N ? g.work[at] : at; }

template <typename T, int HD> struct Rows {
    static constexpr int NB = HD / 16;
    const T* base;
    uint32_t pitch, col;       // values; col: of this lane's first value in a row operand
    __device__ __forceinline__ Rows(const void* p, int64_t pitch_, int64_t col0) : base(static_cast<const T*>(p) + col0), pitch((uint32_t)pitch_) {
        col = ((threadIdx.x & 63) >> 4) * 4;
    }
    // row operand of token voxel v: lane (row, slots 4 (l / 16) + j)
    __device__ __forceinline__ void row(uint32_t v, Frag<T> (&f)[NB]) const {
#pragma unroll
        for (int b = 0; b < NB; ++b) f[b].load(base + (__umul24(v, pitch) + col + b * 16));
    }
    // fp32 column operand: lane (channel 16 b + l % 16, slots = the tokens 4 (l / 16) + j with voxels v[j])
    __device__ __forceinline__ void column(const int (&v)[4], const Frag<T> (&rows)[NB], Frag<float> (&f)[NB], bool careful) const {
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int j = 0; j < 4; ++j) f[b].v[j] = base[__umul24((uint32_t)v[j], pitch) + b * 16 + (threadIdx.x & 15)];
        } else {
            // the row operand turned and widened on the matrix core: a product with the identity, exact for 16-bit values
            f32x4 one;
#pragma unroll
            for (int j = 0; j < 4; ++j) one[j] = (int)(((threadIdx.x & 63) >> 4) * 4 + j) == (int)(threadIdx.x & 15) ? 1.f : 0.f;
            const Frag<T> id = packed<T>(one);
#pragma unroll
            for (int b = 0; b < NB; ++b) f[b].v = mma(rows[b], id, f32x4{0.f, 0.f, 0.f, 0.f});
            if (careful) {                                               // the product spreads what is not finite over its row
                const int l16 = threadIdx.x & 15, quad = (threadIdx.x & 63) >> 4;
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const uint2 w = __builtin_bit_cast(uint2, rows[b].v);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int from = (l16 >> 2) * 16 + quad * 4 + j; // holds channels 4 (l16 / 4) .. + 3 of token 4 quad + j
                        const uint32_t lo = __shfl(w.x, from, 64), hi = __shfl(w.y, from, 64), pair = l16 & 2 ? hi : lo;
                        f[b].v[j] = to_acc(__builtin_bit_cast(T, (uint16_t)(l16 & 1 ? pair >> 16 : pair)));
                    }
                }
            }
        }
    }
    // clears the slots behind the window's end: they hold its last token again, with P = 0
    static __device__ __forceinline__ void clear(int last, Frag<float> (&f)[NB]) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j) f[b].v[j] = (int)((threadIdx.x & 63) >> 4) * 4 + j > last ? 0.f : f[b].v[j];
    }
};

// What a step of 16 tokens needs before their rows can be read: the voxel of this lane's row, and the voxels and words of the
// four tokens in this lane's reduction slots.  Requested a step ahead.  Full steps (all but a window's last) read 16 bytes.
template <typename T> struct Step {
    int row;
    int v[4];
    uint32_t w[4];
    __device__ __forceinline__ void load(const Args& g, int r0, int to) {
        const int l16 = threadIdx.x & 15, quad = (threadIdx.x & 63) >> 4, last = to - 1 - r0;
        row = g.order[r0 + min(l16, last)];
        if (last >= 15) {
            const u32x4_any x = *reinterpret_cast<const u32x4_any*>(g.word + r0 + quad * 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = x[j];
            if (sizeof(T) == 4) {
                const u32x4_any y = *reinterpret_cast<const u32x4_any*>(g.order + r0 + quad * 4);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = (int)y[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = r0 + min(quad * 4 + j, last);
                w[j] = g.word[r];
                if (sizeof(T) == 4) v[j] = g.order[r];
            }
        }
    }
};

// the head's bias table, in units of log 2
__device__ __forceinline__ void stage_table(const Args& g, int h, float* table) {
    for (int i = threadIdx.x; i < g.rows; i += WAVES * 64) table[i] = g.table[(int64_t)i * g.H + h] * LOG2E;
    __syncthreads();
}

// A score in units of log 2, less what the accumulator started from: product + bias, and where a window has several mask
// regions the mask; other windows of a merged block do not take part.
template <bool FAST>
__device__ __forceinline__ float score(float acc, float scale2, uint32_t pq, uint32_t pk, const float* table) {
    const uint32_t d = pq - pk;
    float x = fmaf(acc, scale2, *reinterpret_cast<const float*>(reinterpret_cast<const char*>(table) + (d & 0x7ffcu)));
    if (!FAST && d >> 15) x = (pq ^ pk) >> 23 ? -INFINITY : x + MASKED;
    return x;
}

// ------------------------------------------------------------------------------------------
// forward: own = queries.  fp32: three wavefronts per SIMD, which heads of 32 channels miss by one register (two are spilled;
// 84 742 tokens, windows of 7^3, 3 heads of 32: 74.7 us)
// ------------------------------------------------------------------------------------------
template <typename T, int HD>
__global__ __launch_bounds__(WAVES * 64, sizeof(T) == 4 ? 3 : 1) void flash_forward_kernel(Args g, int64_t groups) {
    constexpr int NB = HD / 16;
    extern __shared__ float table[];
    int h;
    int64_t first;
    place(g.H, groups, h, first);
    const int lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    const int64_t chunk = chunk_of(g, first + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    Blocks blocks(g, chunk * 32 < g.N ? chunk : 0);
    stage_table(g, h, table);
    if (chunk * 32 >= g.N) return;
    blocks.begin(g);
    const int64_t D = (int64_t)g.H * HD;
    const Rows<T, HD> q_rows(g.qkv, 3 * D, h * HD), k_rows(g.qkv, 3 * D, D + h * HD), v_rows(g.qkv, 3 * D, 2 * D + h * HD);
    const float scale2 = g.scale * LOG2E, unscale = 1.f / scale2;
    Block b;
    while (blocks.next(b)) {
        const int subs = (b.len + 15) >> 4;
        Frag<T> q[2][NB];
        uint32_t pq[2];
        int vq[2];
        float offset[2] = {0.f, 0.f}, sum[2] = {0.f, 0.f}, top[2] = {-INFINITY, -INFINITY};
        f32x4 o[2][NB];
        Step<T> ahead;
        ahead.load(g, b.from, b.to);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            vq[s] = __shfl(blocks.voxel, blocks.slot(b, s), 64);
            pq[s] = __shfl(blocks.word, blocks.slot(b, s), 64) + (uint32_t)g.offset4;
#pragma unroll
            for (int c = 0; c < NB; ++c) o[s][c] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const bool general = b.merged || __builtin_amdgcn_readfirstlane(pq[0]) >> 31;   // not one window of one mask region
#pragma unroll
        for (int s = 0; s < 2; ++s) q_rows.row((uint32_t)vq[s], q[s]);
        Frag<T> k_next[NB], v_next[NB];                                  // rows a step ahead, voxels and words two
        uint32_t w_next[4];
        auto request = [&]() {
            k_rows.row((uint32_t)ahead.row, k_next);
            if constexpr (sizeof(T) == 4) v_rows.column(ahead.v, v_next, v_next, false);
            else v_rows.row((uint32_t)ahead.row, v_next);
#pragma unroll
            for (int j = 0; j < 4; ++j) w_next[j] = ahead.w[j];
        };
        request();
        if (b.to - b.from > 16) ahead.load(g, b.from + 16, b.to);
        for (int k0 = b.from; k0 < b.to; k0 += 16) {
            const int last = b.to - 1 - k0;
            Frag<T> k[NB], v[NB];
            Frag<float> vt[NB];
            uint32_t pk[4];
#pragma unroll
            for (int c = 0; c < NB; ++c) k[c] = k_next[c], v[c] = v_next[c];
#pragma unroll
            for (int j = 0; j < 4; ++j) pk[j] = w_next[j];
            if (last >= 16) request();
            if (last >= 32) ahead.load(g, k0 + 32, b.to);
            if constexpr (sizeof(T) == 4) {
#pragma unroll
                for (int c = 0; c < NB; ++c) vt[c] = v[c];
            } else {
                const int none[4] = {0, 0, 0, 0};
                v_rows.column(none, v, vt, blocks.careful);
            }
            if (blocks.careful && last < 15) v_rows.clear(last, vt);
            auto tile = [&](auto fast_tag) {
                constexpr bool FAST = decltype(fast_tag)::value;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (s >= subs) break;
                    const float from = -offset[s] * unscale;             // the accumulator starts at minus the offset
                    f32x4 acc = {from, from, from, from};
#pragma unroll
                    for (int c = 0; c < NB; ++c) acc = mma(k[c], q[s][c], acc);
                    float x[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        x[j] = score<FAST>(acc[j], scale2, pq[s], pk[j], table);
                        if (!FAST && quad * 4 + j > last) x[j] = -INFINITY;
                    }
                    const float xm = fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), before = top[s];
                    top[s] = fmaxf(before, xm);
                    if (!FAST || k0 == b.from || __any(xm > 10.f)) {     // the first tokens; later only by chance
                        const float m = across(xm, true);
                        const bool fresh = across(before, true) == -INFINITY;
                        const float by = m == -INFINITY ? 0.f : fresh ? m : fmaxf(0.f, m), f = fresh ? 0.f : __builtin_amdgcn_exp2f(-by);
                        offset[s] += by;
                        top[s] -= by;
                        sum[s] *= f;
#pragma unroll
                        for (int c = 0; c < NB; ++c) o[s][c] *= f;
#pragma unroll
                        for (int j = 0; j < 4; ++j) x[j] -= by;
                    }
                    f32x4 p;
#pragma unroll
                    for (int j = 0; j < 4; ++j) p[j] = __builtin_amdgcn_exp2f(x[j]);
                    sum[s] += (p[0] + p[1]) + (p[2] + p[3]);
                    const Frag<float> pt = {p};
#pragma unroll
                    for (int c = 0; c < NB; ++c) o[s][c] = mma(vt[c], pt, o[s][c]);
                }
            };
            if (last >= 15 && !general) tile(std::true_type{});
            else tile(std::false_type{});
        }
        if (blocks.again(sum_of(o))) continue;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (s >= subs) break;
            // top: the row's maximum less the offset
            const float z = across(sum[s], false) + 1e-8f * __builtin_amdgcn_exp2f(fmaxf(across(top[s], true), -offset[s]));
            const float inv = 1.f / z;
            if (s * 16 + l16 < b.len) {
                T* row = static_cast<T*>(g.out) + (int64_t)vq[s] * D + h * HD + quad * 4;
#pragma unroll
                for (int c = 0; c < NB; ++c) store4<T>(row + c * 16, o[s][c] * inv);
                if (quad == 0) g.lse[h * g.N + b.a + s * 16 + l16] = offset[s] + __builtin_amdgcn_logf(z);
            }
        }
    }
}

// ------------------------------------------------------------------------------------------
// backward, own = queries: D = dO . O, dQ = scale dS K, where nobody asks for dS
// ------------------------------------------------------------------------------------------
template <typename T, int HD>
__global__ __launch_bounds__(WAVES * 64) void flash_backward_q_kernel(Args g, int64_t groups) {
    constexpr int NB = HD / 16;
    extern __shared__ float table[];
    int h;
    int64_t first;
    place(g.H, groups, h, first);
    const int lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    const int64_t chunk = chunk_of(g, first + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    Blocks blocks(g, chunk * 32 < g.N ? chunk : 0);
    stage_table(g, h, table);
    if (chunk * 32 >= g.N) return;
    blocks.begin(g);
    const int64_t D = (int64_t)g.H * HD;
    const Rows<T, HD> q_rows(g.qkv, 3 * D, h * HD), k_rows(g.qkv, 3 * D, D + h * HD), v_rows(g.qkv, 3 * D, 2 * D + h * HD);
    const Rows<T, HD> do_rows(g.dout, D, h * HD), o_rows(g.out, D, h * HD);
    const float scale2 = g.scale * LOG2E, unscale = 1.f / scale2;
    Block b;
    while (blocks.next(b)) {
        const int subs = (b.len + 15) >> 4;
        Frag<T> q[2][NB], d_o[2][NB];
        uint32_t pq[2];
        int vq[2];
        float lse[2], delta[2];
        f32x4 dq[2][NB];
        Step<T> ahead;
        ahead.load(g, b.from, b.to);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int r = b.a + min(s * 16 + l16, b.len - 1);
            vq[s] = __shfl(blocks.voxel, blocks.slot(b, s), 64);
            pq[s] = __shfl(blocks.word, blocks.slot(b, s), 64) + (uint32_t)g.offset4;
            lse[s] = g.lse[h * g.N + r];
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            Frag<T> o[NB];
            q_rows.row((uint32_t)vq[s], q[s]);
            do_rows.row((uint32_t)vq[s], d_o[s]);
            o_rows.row((uint32_t)vq[s], o);
            float dot = 0.f;
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                dq[s][c] = f32x4{0.f, 0.f, 0.f, 0.f};
                const T* x = reinterpret_cast<const T*>(&d_o[s][c].v);
                const T* y = reinterpret_cast<const T*>(&o[c].v);
#pragma unroll
                for (int j = 0; j < 4; ++j) dot = fmaf(to_acc(x[j]), to_acc(y[j]), dot);
            }
            delta[s] = across(dot, false);
            if (quad == 0 && s * 16 + l16 < b.len) g.delta[h * g.N + b.a + s * 16 + l16] = delta[s];
        }
        const bool general = b.merged || __builtin_amdgcn_readfirstlane(pq[0]) >> 31;   // not one window of one mask region
        for (int k0 = b.from; k0 < b.to; k0 += 16) {
            const int last = b.to - 1 - k0;
            const Step<T> step = ahead;
            Frag<T> k[NB], v[NB];
            Frag<float> kt[NB];
            k_rows.row((uint32_t)step.row, k);
            v_rows.row((uint32_t)step.row, v);
            k_rows.column(step.v, k, kt, blocks.careful);
            if (blocks.careful && last < 15) k_rows.clear(last, kt);
            if (last >= 16) ahead.load(g, k0 + 16, b.to);
            auto tile = [&](auto fast_tag) {
                constexpr bool FAST = decltype(fast_tag)::value;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (s >= subs) break;
                    // the accumulators start at minus the row's log-sum-exp and minus its dO . O
                    const float a0 = -lse[s] * unscale, d0 = -delta[s];
                    f32x4 acc = {a0, a0, a0, a0}, dp = {d0, d0, d0, d0}, ds;
#pragma unroll
                    for (int c = 0; c < NB; ++c) acc = mma(k[c], q[s][c], acc), dp = mma(v[c], d_o[s][c], dp);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float x = score<FAST>(acc[j], scale2, pq[s], step.w[j], table);
                        ds[j] = __builtin_amdgcn_exp2f(x) * dp[j];
                        if (!FAST && quad * 4 + j > last) ds[j] = 0.f;
                    }
                    const Frag<float> dst = {ds};
#pragma unroll
                    for (int c = 0; c < NB; ++c) dq[s][c] = mma(kt[c], dst, dq[s][c]);
                }
            };
            if (last >= 15 && !general) tile(std::true_type{});
            else tile(std::false_type{});
        }
        if (blocks.again(sum_of(dq))) continue;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (s * 16 + l16 < b.len) {
                T* row = static_cast<T*>(g.dqkv) + (int64_t)vq[s] * 3 * D + h * HD + quad * 4;
#pragma unroll
                for (int c = 0; c < NB; ++c) store4<T>(row + c * 16, dq[s][c] * g.scale);
            }
        }
    }
}

// ------------------------------------------------------------------------------------------
// backward from a stored dS: D = dO . O in front of the key side, dQ = scale dS K behind it
// ------------------------------------------------------------------------------------------
template <typename T, int HD> __global__ __launch_bounds__(256) void flash_delta_kernel(Args g) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;           // heads of a token side by side
    if (i >= g.N * g.H) return;
    const int64_t r = i / g.H, h = i - r * g.H, at = ((int64_t)g.order[r] * g.H + h) * HD;
    const T* const a = static_cast<const T*>(g.dout) + at;
    const T* const b = static_cast<const T*>(g.out) + at;
    Frag<T> x[HD / 4], y[HD / 4];
#pragma unroll
    for (int q = 0; q < HD / 4; ++q) x[q].load(a + q * 4), y[q].load(b + q * 4);
    float part[4] = {0.f, 0.f, 0.f, 0.f};                                // summed as four lanes of the query side would
#pragma unroll
    for (int q = 0; q < HD / 4; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            part[q & 3] = fmaf(to_acc(reinterpret_cast<const T*>(&x[q].v)[j]), to_acc(reinterpret_cast<const T*>(&y[q].v)[j]), part[q & 3]);
    g.delta[h * g.N + r] = (part[0] + part[1]) + (part[2] + part[3]);
}

// own = queries
template <typename T, int HD>
__global__ __launch_bounds__(WAVES * 64) void flash_dq_kernel(Args g, int64_t groups) {
    constexpr int NB = HD / 16;
    int h;
    int64_t first;
    place(g.H, groups, h, first);
    const int lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    const int64_t chunk = chunk_of(g, first + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    if (chunk * 32 >= g.N) return;
    Blocks blocks(g, chunk);
    blocks.begin(g);
    const int64_t D = (int64_t)g.H * HD;
    const Rows<T, HD> k_rows(g.qkv, 3 * D, D + h * HD);
    Block b;
    while (blocks.next(b)) {
        int vq[2];
        uint32_t at[2];        // first value of the query's row of dS, less its window's first rank (modulo 2^32: places are below 2^31)
        f32x4 dq[2][NB];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int r = b.a + min(s * 16 + l16, b.len - 1), c = __shfl(blocks.c, blocks.slot(b, s), 64), T0 = __shfl(blocks.T, blocks.slot(b, s), 64);
            vq[s] = __shfl(blocks.voxel, blocks.slot(b, s), 64);
            at[s] = (uint32_t)(g.tok_sq[r] * g.H + h * c * c + (r - T0) * c) - (uint32_t)T0;
#pragma unroll
            for (int c2 = 0; c2 < NB; ++c2) dq[s][c2] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        // 32 keys at a time, whole lines of dS, the next 32 in flight
        struct Tile {
            f32x4 ds[2][2];
            Frag<T> k[2][NB];                                            // 16 bits: rows, fp32: columns
        };
        struct Keys {
            int v[2][sizeof(T) == 4 ? 4 : 1];                            // voxels of the lane's slots, or of its row
        };
        auto keys = [&](int k0, Keys& t) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < (sizeof(T) == 4 ? 4 : 1); ++j) t.v[i][j] = g.order[min(k0 + i * 16 + (sizeof(T) == 4 ? quad * 4 + j : l16), b.to - 1)];
        };
        auto request = [&](int k0, const Keys& from, Tile& t) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if constexpr (sizeof(T) == 4) k_rows.column(from.v[i], t.k[i], t.k[i], false);
                else k_rows.row((uint32_t)from.v[i][0], t.k[i]);
            }
            if (b.to - k0 >= 32 && !b.merged) {
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int i = 0; i < 2; ++i) t.ds[i][s] = *reinterpret_cast<const f32x4_any*>(g.ds + (at[s] + (uint32_t)(k0 + i * 16 + quad * 4)));
            } else {                                                     // the window's own tokens
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const int T0 = __shfl(blocks.T, blocks.slot(b, s), 64), end = T0 + __shfl(blocks.c, blocks.slot(b, s), 64);
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const int r = k0 + i * 16 + quad * 4 + j;
                            t.ds[i][s][j] = r >= T0 && r < end ? g.ds[at[s] + (uint32_t)r] : 0.f;
                        }
                }
            }
        };
        Tile tile;
        Keys next;
        keys(b.from, next);
        request(b.from, next, tile);
        if (b.to - b.from > 32) keys(b.from + 32, next);
        for (int k0 = b.from; k0 < b.to; k0 += 32) {
            const Tile now = tile;
            if (b.to - k0 > 32) request(k0 + 32, next, tile);
            if (b.to - k0 > 64) keys(k0 + 64, next);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int last = b.to - 1 - k0 - i * 16;
                if (last < 0) break;
                Frag<float> kt[NB];
                if constexpr (sizeof(T) == 4) {
#pragma unroll
                    for (int c = 0; c < NB; ++c) kt[c] = now.k[i][c];
                } else {
                    const int none[4] = {0, 0, 0, 0};
                    k_rows.column(none, now.k[i], kt, blocks.careful);
                }
                if (blocks.careful && last < 15) k_rows.clear(last, kt);
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const Frag<float> ds = {now.ds[i][s]};
#pragma unroll
                    for (int c = 0; c < NB; ++c) dq[s][c] = mma(kt[c], ds, dq[s][c]);
                }
            }
        }
        if (blocks.again(sum_of(dq))) continue;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (s * 16 + l16 < b.len) {
                T* row = static_cast<T*>(g.dqkv) + (int64_t)vq[s] * 3 * D + h * HD + quad * 4;
#pragma unroll
                for (int c = 0; c < NB; ++c) store4<T>(row + c * 16, dq[s][c] * g.scale);
            }
        }
    }
}

// ------------------------------------------------------------------------------------------
// backward, own = keys: dV = P^T dO, dK = scale dS^T Q; STORE: dS for the bias gradient and for dQ
// ------------------------------------------------------------------------------------------
template <typename T, int HD, bool STORE>
__global__ __launch_bounds__(WAVES * 64) void flash_backward_kv_kernel(Args g, int64_t groups) {
    constexpr int NB = HD / 16;
    extern __shared__ float table[];
    int h;
    int64_t first;
    place(g.H, groups, h, first);
    const int lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4;
    const int64_t chunk = chunk_of(g, first + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    Blocks blocks(g, chunk * 32 < g.N ? chunk : 0);
    stage_table(g, h, table);
    if (chunk * 32 >= g.N) return;
    blocks.begin(g);
    const int64_t D = (int64_t)g.H * HD;
    const Rows<T, HD> q_rows(g.qkv, 3 * D, h * HD), k_rows(g.qkv, 3 * D, D + h * HD), v_rows(g.qkv, 3 * D, 2 * D + h * HD);
    const Rows<T, HD> do_rows(g.dout, D, h * HD);
    const float scale2 = g.scale * LOG2E, unscale = 1.f / scale2;
    Block b;
    while (blocks.next(b)) {
        const int subs = (b.len + 15) >> 4;
        Frag<T> k[2][NB], v[2][NB];
        uint32_t pk[2];
        int vk[2];
        uint32_t at[2];        // first value of the key's column of dS, less its window's first rank times the row's length
        int width[2];          // of a row of dS
        f32x4 dk[2][NB], dv[2][NB];
        Step<T> ahead;
        ahead.load(g, b.from, b.to);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            vk[s] = __shfl(blocks.voxel, blocks.slot(b, s), 64);
            pk[s] = __shfl(blocks.word, blocks.slot(b, s), 64);
            if constexpr (STORE) {
                const int r = b.a + min(s * 16 + l16, b.len - 1), T0 = __shfl(blocks.T, blocks.slot(b, s), 64);
                width[s] = __shfl(blocks.c, blocks.slot(b, s), 64);
                at[s] = (uint32_t)(g.tok_sq[r] * g.H + h * width[s] * width[s] + r - T0) - (uint32_t)T0 * (uint32_t)width[s];
            }
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            k_rows.row((uint32_t)vk[s], k[s]);
            v_rows.row((uint32_t)vk[s], v[s]);
#pragma unroll
            for (int c = 0; c < NB; ++c) dk[s][c] = dv[s][c] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        const bool general = b.merged || __builtin_amdgcn_readfirstlane(pk[0]) >> 31;
        for (int q0 = b.from; q0 < b.to; q0 += 16) {
            const int last = b.to - 1 - q0;
            const Step<T> step = ahead;
            f32x4 lse, delta;
            if (last >= 15) {
                lse = *reinterpret_cast<const f32x4_any*>(g.lse + h * g.N + q0 + quad * 4);
                delta = *reinterpret_cast<const f32x4_any*>(g.delta + h * g.N + q0 + quad * 4);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int64_t r = h * g.N + q0 + min(quad * 4 + j, last);
                    lse[j] = g.lse[r];
                    delta[j] = g.delta[r];
                }
            }
            Frag<T> q[NB], d_o[NB];
            Frag<float> qt[NB], dot[NB];
            q_rows.row((uint32_t)step.row, q);
            do_rows.row((uint32_t)step.row, d_o);
            q_rows.column(step.v, q, qt, blocks.careful);
            do_rows.column(step.v, d_o, dot, blocks.careful);
            if (blocks.careful && last < 15) {
                q_rows.clear(last, qt);
                do_rows.clear(last, dot);
            }
            if (last >= 16) ahead.load(g, q0 + 16, b.to);
            const f32x4 a0 = lse * -unscale, d0 = -delta;               // what the accumulators start from
            auto tile = [&](auto fast_tag) {
                constexpr bool FAST = decltype(fast_tag)::value;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    if (s >= subs) break;
                    f32x4 acc = a0, dp = d0, p, ds;
#pragma unroll
                    for (int c = 0; c < NB; ++c) acc = mma(q[c], k[s][c], acc), dp = mma(d_o[c], v[s][c], dp);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        p[j] = __builtin_amdgcn_exp2f(score<FAST>(acc[j], scale2, step.w[j] + (uint32_t)g.offset4, pk[s], table));
                        if (!FAST && quad * 4 + j > last) p[j] = 0.f;
                        ds[j] = p[j] * dp[j];
                        if (!FAST && quad * 4 + j > last) ds[j] = 0.f;
                    }
                    if constexpr (STORE) {
                        if (s * 16 + l16 < b.len) {                      // four rows of dS, sixteen neighbours of each per store
                            const uint32_t to = at[s] + (uint32_t)(q0 + quad * 4) * (uint32_t)width[s];
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                if (FAST || (quad * 4 + j <= last && !((pk[s] ^ step.w[j]) >> 23))) g.ds[to + (uint32_t)(j * width[s])] = ds[j];
                        }
                    }
                    const Frag<float> pf = {p}, df = {ds};
#pragma unroll
                    for (int c = 0; c < NB; ++c) dv[s][c] = mma(dot[c], pf, dv[s][c]), dk[s][c] = mma(qt[c], df, dk[s][c]);
                }
            };
            if (last >= 15 && !general) tile(std::true_type{});
            else tile(std::false_type{});
        }
        if (blocks.again(sum_of(dk) + sum_of(dv))) continue;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if (s * 16 + l16 < b.len) {
                T* row = static_cast<T*>(g.dqkv) + (int64_t)vk[s] * 3 * D + h * HD + quad * 4;
#pragma unroll
                for (int c = 0; c < NB; ++c) {
                    store4<T>(row + D + c * 16, dk[s][c] * g.scale);
                    store4<T>(row + 2 * D + c * 16, dv[s][c]);
                }
            }
        }
    }
}

template <typename K> static int launch(K kernel, const Args& g, hipStream_t s, const char* what, bool table = true) {
    const int64_t groups = (g.N + 32 * WAVES - 1) / (32 * WAVES);
    SSWIN_CHECK(groups * g.H < (1ll << 31), "%s: too many tokens", what);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(groups * g.H)), dim3(WAVES * 64), table ? (size_t)g.rows * sizeof(float) : 0, s, g, groups);
    return launch_ok(what);
}

// With dS asked for, the query side reads what the key side has stored instead of forming scores, exponentials and dP again.
template <typename T, int HD> static int launch_backward(const Args& g, hipStream_t s) {
    if (!g.ds) {
        if (int rc = launch(flash_backward_q_kernel<T, HD>, g, s, "flash_backward, queries")) return rc;
        return launch(flash_backward_kv_kernel<T, HD, false>, g, s, "flash_backward, keys");
    }
    hipLaunchKernelGGL((flash_delta_kernel<T, HD>), dim3((unsigned)((g.N * g.H + 255) / 256)), dim3(256), 0, s, g);
    if (int rc = launch_ok("flash_backward, delta")) return rc;
    if (int rc = launch(flash_backward_kv_kernel<T, HD, true>, g, s, "flash_backward, keys")) return rc;
    return launch(flash_dq_kernel<T, HD>, g, s, "flash_backward, queries", false);
}

}  // namespace flash
}  // namespace sswin

using namespace sswin;
using namespace sswin::flash;

static int flash_check(const char* what, int dtype, int64_t N, int H, int hd, int n, int rows, int offset0) {
    SSWIN_CHECK(dtype >= SSWIN_F32 && dtype <= SSWIN_BF16, "%s: value type %d", what, dtype);
    SSWIN_CHECK(N >= 0 && N < MAX_TOKENS && H > 0 && H < 256, "%s: bad sizes", what);
    SSWIN_CHECK(hd == 16 || hd == 32, "%s: heads of %d channels (16 or 32 are supported)", what, hd);
    SSWIN_CHECK(n > 0 && rows > 0 && rows <= MAX_ROWS && offset0 >= 0, "%s: a bias table of at most %d rows", what, MAX_ROWS);
    SSWIN_CHECK(N * 3 * H * hd < (1ll << 32), "%s: token rows need 32-bit offsets", what);
    return 0;
}

extern "C" {

int sswin_flash_supported(int dtype, int64_t N, int H, int hd, int rows) {
    return dtype >= SSWIN_F32 && dtype <= SSWIN_BF16 && N > 0 && N < MAX_TOKENS && (hd == 16 || hd == 32) && rows > 0 && rows <= MAX_ROWS && H > 0 && H < 256 &&
           N * 3 * H * hd < (1ll << 32);
}

// Below, all wavefronts find a place at once (three a SIMD), and above, one workgroup is a while about it and the last places weigh little.
// Words, forward and backward by rank and ordered, us (windows of 7^3, heads of 16; chunks x heads): fp32 1032 77 and 77, 1944 104 and 104, 2040 100 and 91,
// 2964 115 and 111; 3462 147 and 141, 3966 165 and 148, 5940 185 and 157, 6978 188 and 168, 10 569 226 and 209, 13 968 400 and 356, 21 165 483 and 471;
// fp16 1032 64 and 66, 1944 84 and 84, 2040 80 and 75, 2964 93 and 91; 3462 115 and 112, 3966 129 and 118, 5940 146 and 124, 10 569 173 and 161, 21 165 366 and 360.
size_t sswin_flash_order_ints(int64_t N, int H) {
    const int64_t chunks = (N + 31) / 32;
    return chunks <= ORDER_MOST && chunks * H > 12 * (int64_t)device_cus() ? (size_t)chunks : 0;
}

int sswin_flash_tokens_ordered(const int32_t* plan, int64_t g_cap, int64_t groups, const int32_t* tokens, int64_t N, int H, int n, const int32_t* code,
                               const int8_t* mask, int nmw, int32_t* word, int32_t* tok_sq, int32_t* order, void* stream) {
    SSWIN_CHECK(N >= 0 && n > 0 && H > 0 && groups >= 0 && groups <= g_cap && groups % H == 0, "flash_tokens: bad sizes");
    if (N == 0 || groups == 0) return 0;
    SSWIN_CHECK(plan && tokens && code && word && (!mask || nmw > 0), "flash_tokens: null pointer");
    SSWIN_CHECK(!order || (N + 31) / 32 <= ORDER_MOST, "flash_tokens: an order of %lld tokens", (long long)N);
    const int64_t windows = groups / H;
    hipLaunchKernelGGL(flash_tokens_kernel, dim3((unsigned)((windows + TOKENS_WAVES - 1) / TOKENS_WAVES + (order ? 1 : 0))), dim3(ORDER_THREADS), 0,
                       static_cast<hipStream_t>(stream), plan, g_cap, windows, H, tokens + 3 * N, N, code, mask, nmw, n, reinterpret_cast<uint32_t*>(word), tok_sq, order);
    return launch_ok("flash_tokens");
}
int sswin_flash_tokens(const int32_t* plan, int64_t g_cap, int64_t groups, const int32_t* tokens, int64_t N, int H, int n, const int32_t* code,
                       const int8_t* mask, int nmw, int32_t* word, int32_t* tok_sq, void* stream) {
    return sswin_flash_tokens_ordered(plan, g_cap, groups, tokens, N, H, n, code, mask, nmw, word, tok_sq, nullptr, stream);
}

int sswin_flash_forward_ordered(int dtype, const int32_t* tokens, const int32_t* word, const int32_t* order, int64_t N, int H, int hd, int n, const void* qkv,
                                float scale, const float* table, int rows, int offset0, void* out, float* lse, void* stream) {
    if (int rc = flash_check("flash_forward", dtype, N, H, hd, n, rows, offset0)) return rc;
    if (N == 0) return 0;
    SSWIN_CHECK(tokens && word && qkv && table && out && lse, "flash_forward: null pointer");
    SSWIN_CHECK(((uintptr_t)qkv | (uintptr_t)out) % 16 == 0, "flash_forward: pointers must be 16-byte aligned");
    Args g = {};
    g.order = tokens, g.tok_T = tokens + N, g.tok_c = tokens + 2 * N, g.word = reinterpret_cast<const uint32_t*>(word);
    g.N = N, g.H = H, g.rows = rows, g.offset4 = offset0 * 4, g.scale = scale, g.table = table, g.qkv = qkv, g.out = out, g.lse = lse, g.work = order;
    hipStream_t s = static_cast<hipStream_t>(stream);
#define FLASH(K, T) (hd == 16 ? launch(K<T, 16>, g, s, #K) : launch(K<T, 32>, g, s, #K))
    if (dtype == SSWIN_F32) return FLASH(flash_forward_kernel, float);
    if (dtype == SSWIN_F16) return FLASH(flash_forward_kernel, __half);
    return FLASH(flash_forward_kernel, __hip_bfloat16);
#undef FLASH
}

int sswin_flash_forward(int dtype, const int32_t* tokens, const int32_t* word, int64_t N, int H, int hd, int n, const void* qkv, float scale, const float* table,
                        int rows, int offset0, void* out, float* lse, void* stream) {
    return sswin_flash_forward_ordered(dtype, tokens, word, nullptr, N, H, hd, n, qkv, scale, table, rows, offset0, out, lse, stream);
}

int sswin_flash_backward_ordered(int dtype, const int32_t* tokens, const int32_t* word, const int32_t* tok_sq, const int32_t* order, int64_t N, int H, int hd, int n,
                                 const void* qkv, float scale, const float* table, int rows, int offset0, const void* out, const float* lse, const void* dout,
                                 void* dqkv, float* delta, float* ds, void* stream) {
    if (int rc = flash_check("flash_backward", dtype, N, H, hd, n, rows, offset0)) return rc;
    if (N == 0) return 0;
    SSWIN_CHECK(tokens && word && qkv && table && out && lse && dout && dqkv && delta && (!ds || tok_sq), "flash_backward: null pointer");
    SSWIN_CHECK(((uintptr_t)qkv | (uintptr_t)out | (uintptr_t)dout | (uintptr_t)dqkv) % 16 == 0, "flash_backward: pointers must be 16-byte aligned");
    Args g = {};
    g.order = tokens, g.tok_T = tokens + N, g.tok_c = tokens + 2 * N, g.word = reinterpret_cast<const uint32_t*>(word);
    g.N = N, g.H = H, g.rows = rows, g.offset4 = offset0 * 4, g.scale = scale, g.table = table, g.qkv = qkv, g.out = const_cast<void*>(out);
    g.lse = const_cast<float*>(lse), g.dout = dout, g.delta = delta, g.dqkv = dqkv, g.ds = ds, g.tok_sq = tok_sq, g.work = order;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == SSWIN_F32) return hd == 16 ? launch_backward<float, 16>(g, s) : launch_backward<float, 32>(g, s);
    if (dtype == SSWIN_F16) return hd == 16 ? launch_backward<__half, 16>(g, s) : launch_backward<__half, 32>(g, s);
    return hd == 16 ? launch_backward<__hip_bfloat16, 16>(g, s) : launch_backward<__hip_bfloat16, 32>(g, s);
}
int sswin_flash_backward(int dtype, const int32_t* tokens, const int32_t* word, const int32_t* tok_sq, int64_t N, int H, int hd, int n, const void* qkv, float scale,
                         const float* table, int rows, int offset0, const void* out, const float* lse, const void* dout, void* dqkv, float* delta, float* ds,
                         void* stream) {
    return sswin_flash_backward_ordered(dtype, tokens, word, tok_sq, nullptr, N, H, hd, n, qkv, scale, table, rows, offset0, out, lse, dout, dqkv, delta, ds, stream);
}

}  // extern "C"
