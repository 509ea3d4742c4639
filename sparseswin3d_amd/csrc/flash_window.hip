// Window attention for heads of 16 channels in windows of up to 384 positions: a wavefront per (window, head) and up to 96 of the
// window's tokens (WindowAttention.forward, sparse_swin/swin3d_base.py:654-675, from the projected qkv to the attention output, and
// its backward with the gradient of the bias table in the same launch).  flash_attention.hip serves what these do not take: heads of 32
// channels, more positions, heads or windows (sswin_flash_window_list_ints), and windows of a few tokens (sswin_flash_window_faster).
//
// Work: the windows by descending size (flash_window_tokens_kernel), dealt to as many workgroups as find a place at once; a workgroup keeps a
// head's bias table, and in the backward the sums of its gradient, in LDS.  A window of up to KT tiles of 16 tokens is one wavefront's, one
// of up to 2 KT tiles two wavefronts', larger ones take a workgroup of four.  All products are 16 x 16 tiles, laid out as in
// flash_attention.hip: an accumulator is the operand of the next product over its rows.
//
// What this changes against blocks of 32 keys (flash_attention.hip): the scores of a window are formed once in the backward, not dS stored for dQ and for
// the table's gradient (217 MB written and read twice with 225 700 tokens); rows are read once a window instead of once a block; P and dS meet
// rows on the 16-bit matrix cores.  The table's gradient is summed by 64-bit integer additions in LDS, which take 10 clocks a wavefront's 64
// (floating-point ones 180: what kept the sums out of the backward), and whose result does not depend on their order.
//
// Windows of 7^3, 3 heads of 16, a call with all its launches (words, D, sums), us, chunks of 32 tokens -> here: 112 700 tokens fp32 forward 63 -> 56, backward with the
// table's gradient 222 -> 115; 225 700 fp16 83 -> 68 and 361 -> 153; 8100 tokens in 50 windows of 12 to 316, 24 heads: fp32 68 -> 81 and 257 -> 163, fp16 55 -> 68 and
// 189 -> 138 (a forward of so few large windows has one workgroup for each, whose first wavefronts walk over the keys twice; training and inference take the same
// kernels, for the same bits).  Half of the time a SIMD of the backward issues vector instructions (fp32 990 clocks of 1950 a tile, fp16 720 of 1340: 225 700 tokens), the
// matrix cores are busy 160 and 96 clocks: two wavefronts a SIMD, held there by their registers (fp32 all 256 with 20 more and 109 scalar ones spilled, 16 bit 236 with 92
// to 101 scalar ones), wait for each other's rows, transpositions and exponentials.
#include "flash_window.hpp"

namespace sswin {
namespace flash {
namespace window {

constexpr int KT = MOST / WAVES;                                         // tiles of 16 tokens of a wavefront in the backward

// The windows by descending number of tiles, by one workgroup, and the word of every token, a wavefront per window.
__device__ __forceinline__ void order_windows(const int32_t* __restrict__ plan, int windows, int H, int32_t* __restrict__ list) {
    __shared__ uint16_t place[MOST * LIST_THREADS];                      // [class, most tiles first][thread]
    __shared__ int sums[LIST_THREADS / 64];
    const int t = threadIdx.x, per = (windows + LIST_THREADS - 1) / LIST_THREADS, begin = min(t * per, windows), end = min(begin + per, windows);
    auto kind = [&](int k) { return MOST - max(1, min((plan[(int64_t)k * H] + 15) >> 4, MOST)); };
    for (int k = 0; k < MOST; ++k) place[k * LIST_THREADS + t] = 0;
    for (int k = begin; k < end; ++k) ++place[kind(k) * LIST_THREADS + t];
    __syncthreads();
    // sums in front, classes first; a thread adds MOST neighbours
    int own = 0;
    for (int k = 0; k < MOST; ++k) own += place[t * MOST + k];
    int before = own;
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(before, o, 64);
        if ((t & 63) >= o) before += v;
    }
    if ((t & 63) == 63) sums[t >> 6] = before;
    __syncthreads();
    before -= own;
    for (int w = 0; w < t >> 6; ++w) before += sums[w];
    for (int k = 0; k < MOST; ++k) {
        const int n = place[t * MOST + k];
        place[t * MOST + k] = (uint16_t)before;
        before += n;
    }
    __syncthreads();
    // windows of more than t tiles: those in front of the class of t tiles
    if (t < LIST_HEAD) list[t] = t >= MOST ? 0 : t == 0 ? windows : place[(MOST - t) * LIST_THREADS];
    __syncthreads();
    for (int k = begin; k < end; ++k) list[LIST_HEAD + place[kind(k) * LIST_THREADS + t]++] = k;
}

__global__ __launch_bounds__(LIST_THREADS) void flash_window_tokens_kernel(const int32_t* __restrict__ plan, int64_t g_cap, int windows, int H,
                                                                           const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ code,
                                                                           const int8_t* __restrict__ mask, int nmw, int n, uint32_t* __restrict__ word,
                                                                           int32_t* __restrict__ list) {
    if (blockIdx.x == 0) return order_windows(plan, windows, H, list);
    const int k = (int)(blockIdx.x - 1) * (LIST_THREADS / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (k >= windows) return;
    const int64_t g = (int64_t)k * H;                                    // the window's first group (head 0)
    const int c = plan[g], T = plan[g_cap + g], w = plan[3 * g_cap + g], lane = threadIdx.x & 63;
    const int8_t* region = mask ? mask + (int64_t)(w % nmw) * n : nullptr;
    int low = 1 << 30;                                                   // words hold codes from zero on
    for (int i = lane; i < n; i += 64) low = min(low, code[i]);
    for (int o = 1; o < 64; o <<= 1) low = min(low, __shfl_xor(low, o, 64));
    uint32_t several = 0;
    if (region) {
        const int8_t r0 = region[tok_pos[T]];
        bool differ = false;
        for (int i = lane; i < c; i += 64) differ = differ || region[tok_pos[T + i]] != r0;
        several = __any(differ) ? 0x80000000u : 0u;
    }
    for (int i = lane; i < c; i += 64) {
        const int p = tok_pos[T + i];
        word[T + i] = (uint32_t)(code[p] - low) * 4u | (region ? ((uint32_t)(uint8_t)region[p]) << 15 : 0u) | several;
    }
}

// What a wavefront multiplies with P or dS: rows turned, 16-bit tokens one piece, fp32 tokens two
template <typename T> struct Column {
    f16x8 h;
    __device__ __forceinline__ void set(const f32x4& x) { h = with_rest(halves(x)); }
    __device__ __forceinline__ f32x4 times(const Fine& p, const f32x4& c) const { return mma32(h, both(p), c); }
};
template <> struct Column<float> {
    f16x8 h, l;
    __device__ __forceinline__ void set(const f32x4& v) {
        const Pair x = split(v);
        h = with_rest(x.h), l = with_rest(x.l);
    }
    __device__ __forceinline__ f32x4 times(const Fine& p, const f32x4& c) const { return mma32(l, both(p), mma32(h, both(p), c)); }
};
// The same held for a whole window, in half the registers: the parts of a sum, the second in units of 1 / REST
struct Sum {
    f32x4 a, b;
    __device__ __forceinline__ f32x4 total() const { return a + b * (1.f / REST); }
};
template <typename T> struct Held {
    f16x4 h;
    __device__ __forceinline__ void set(const f32x4& x) { h = halves(x); }
    __device__ __forceinline__ void add(const Fine& p, Sum& s) const { s.a = mma16(h, p.h, s.a), s.b = mma16(h, p.l, s.b); }
};
template <> struct Held<float> {
    Fine x;
    __device__ __forceinline__ void set(const f32x4& v) { x = split_fine(v); }
    __device__ __forceinline__ void add(const Fine& p, Sum& s) const { s.a = mma16(x.h, p.h, s.a), s.b = mma32(both(x.h, x.l), both(p.l, p.h), s.b); }
};

// ------------------------------------------------------------------------------------------
// forward: a wavefront holds the queries of its tiles and walks over the window's keys, 16 at a time
// ------------------------------------------------------------------------------------------
constexpr int F_TILES = 4;                                               // tiles of queries of a wavefront at a time
// Wavefronts a SIMD.  Three and four at 16 bit, with the words, us: 112 700 tokens fp16 47.5 and 41.5, bf16 46 and 43; 225 700 75.4 and 73.1, 76 and 72.4; 8100 in nearly
// full windows the same (24 bytes a lane of the fp16 kernel spilled); fp32 needs 149 registers.
constexpr int forward_resident(size_t value) { return value == 4 ? 3 : 4; }

template <typename T> __global__ __launch_bounds__(WAVES * 64, forward_resident(sizeof(T))) void flash_window_forward_kernel(Args g) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* const turn = reinterpret_cast<float*>(lds) + wave * TURN;
    float* const bias = reinterpret_cast<float*>(lds) + WAVES * TURN;
    const uint32_t bias_at = lds_address(bias);
    int h, first;
    place(g.H, h, first);
    Work<F_TILES> work(g, first);
    stage_table(g, h, bias);
    __syncthreads();
    const int D = g.H * HD;
    const Rows<T> q_rows(g.qkv, g.N, 3 * D, h * HD), k_rows(g.qkv, g.N, 3 * D, D + h * HD), v_rows(g.qkv, g.N, 3 * D, 2 * D + h * HD), o_rows(g.out, g.N, D, h * HD);
    const Buffer order = buffer(g.order, g.N), word = buffer(g.word, g.N);
    constexpr bool HALVES = std::is_same<T, __half>::value;
    const float scale2 = g.scale * LOG2E, unscale = 1.f / scale2;
    float most = 0.f;
    // F_TILES tiles of queries from tile `from` on; MASK: windows of several mask regions
    auto run = [&](int c, int T0, int from, int count, auto masked_tag) __attribute__((always_inline)) {
        constexpr bool MASK = decltype(masked_tag)::value;
        constexpr uint32_t KEPT = MASK ? 0x7fffffffu : INDEX;            // of a word
        const int all = (c + 15) >> 4;
        struct Strip {                                                   // 16 keys
            Frag<T> k, v;
            u32x4 w;
        };
        auto voxel_of = [&](int s) { return (int)load1(order, l16 * 4, (T0 + s * 16) * 4); };
        auto request = [&](int s, int voxel, Strip& x) {
            k_rows.row(voxel, x.k);
            v_rows.row(voxel, x.v);
            x.w = load4(word, quad * 16, (T0 + s * 16) * 4);
        };
        Frag<T> q[F_TILES];
        uint32_t pq[F_TILES];
        int vq[F_TILES];
        float offset[F_TILES], sum[F_TILES], top[F_TILES];
        f32x4 o[F_TILES];
        int voxel_ahead = voxel_of(0);
#pragma unroll
        for (int t = 0; t < F_TILES; ++t) {
            offset[t] = sum[t] = 0.f, top[t] = -INFINITY;
            o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
            vq[t] = load1(order, l16 * 4, (T0 + (from + t) * 16) * 4);   // behind the window's end: some other token
            pq[t] = (load1(word, l16 * 4, (T0 + (from + t) * 16) * 4) & KEPT) + (uint32_t)g.offset4 + (MASK ? 0 : bias_at);
        }
        Strip ahead;
        request(0, voxel_ahead, ahead);
        if (all > 1) voxel_ahead = voxel_of(1);
#pragma unroll
        for (int t = 0; t < F_TILES; ++t) q_rows.row(vq[t], q[t]);
#pragma clang loop unroll(disable)
        for (int s = 0; s < all; ++s) {
            Strip now = ahead;
            if (s + 1 < all) request(s + 1, voxel_ahead, ahead);
            if (s + 2 < all) voxel_ahead = voxel_of(s + 2);
            const int last = c - 1 - s * 16;
            keep(l16 <= last, now.k), keep(l16 <= last, now.v);          // nothing behind the window's end
            u32x4 wk;
#pragma unroll
            for (int j = 0; j < 4; ++j) wk[j] = now.w[j] & KEPT;
            const f32x4 vw = widened(now.v);
            most = fmaxf(most, largest_finite(vw));
            const Frag<float> vt = {turned(turn, vw)};
            // fp16 tokens: V is a piece as it is and P two, one product of 16 clocks where fp32 takes 128 (three wavefronts a SIMD, 225 700 tokens with the words 79.7 -> 73.5 us,
            // 37 200 in 6 heads 42.0 -> 39.5).  P is at most 2^10 and keeps 22 bits, or 2^-36, of which a result of 11 bits shows nothing.  The second piece of P may be zero
            // or negative: infinities meet P itself.
            Column<T> vh;
            bool plain = false;
            if constexpr (HALVES) {
                const float odd = not_finite(vw);
                vh.set(vt.v), plain = !__any(odd != odd);
            }
            auto tiles = [&](auto from_tag, auto count_tag) __attribute__((always_inline)) {
                constexpr int FROM = decltype(from_tag)::value, COUNT = decltype(count_tag)::value;   // two at a time: one's exponentials beside the other's products
                float x[COUNT][4], xm[COUNT];
                bool over = false;
#pragma unroll
                for (int i = 0; i < COUNT; ++i) {
                    const int t = FROM + i;
                    const float start = -offset[t] * unscale;            // the accumulator starts at minus the offset
                    f32x4 acc = {start, start, start, start};
                    acc = mma(now.k, q[t], acc);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t d = pq[t] - wk[j];
                        x[i][j] = fmaf(acc[j], scale2, lds_float(MASK ? (d & INDEX) + bias_at : d));
                        if (MASK && d >> 15) x[i][j] += MASKED;
                    }
                    if (last < 15) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) x[i][j] = quad * 4 + j > last ? -INFINITY : x[i][j];
                    }
                    xm[i] = fmaxf(fmaxf(x[i][0], x[i][1]), fmaxf(x[i][2], x[i][3]));
                    over = over || xm[i] > 10.f;
                }
                const bool move = s == 0 || __any(over);                 // the first tokens; later only by chance
#pragma unroll
                for (int i = 0; i < COUNT; ++i) {
                    const int t = FROM + i;
                    const float before = top[t];
                    top[t] = fmaxf(before, xm[i]);
                    if (move) {
                        const float m = across_max(xm[i]);
                        const bool fresh = across_max(before) == -INFINITY;
                        const float by = m == -INFINITY ? 0.f : fresh ? m : fmaxf(0.f, m), f = fresh ? 0.f : __builtin_amdgcn_exp2f(-by);
                        offset[t] += by;
                        top[t] -= by;
                        sum[t] *= f;
                        o[t] *= f;
#pragma unroll
                        for (int j = 0; j < 4; ++j) x[i][j] -= by;
                    }
                    f32x4 p;
#pragma unroll
                    for (int j = 0; j < 4; ++j) p[j] = __builtin_amdgcn_exp2f(x[i][j]);
                    sum[t] += (p[0] + p[1]) + (p[2] + p[3]);
                    if constexpr (HALVES) {
                        if (plain) o[t] = vh.times(split_fine(p), o[t]);
                        else o[t] = mma(Frag<float>{widened(Frag<__half>{__builtin_shufflevector(vh.h, vh.h, 0, 1, 2, 3)})}, Frag<float>{p}, o[t]);
                    } else {
                        o[t] = mma(vt, Frag<float>{p}, o[t]);
                    }
                }
            };
            auto two = [&](auto from_tag) __attribute__((always_inline)) {
                const int more = count - decltype(from_tag)::value;
                if (more > 1) tiles(from_tag, std::integral_constant<int, 2>{});
                else if (more > 0) tiles(from_tag, std::integral_constant<int, 1>{});
            };
            two(std::integral_constant<int, 0>{});
            two(std::integral_constant<int, 2>{});
        }
#pragma unroll
        for (int t = 0; t < F_TILES; ++t) {
            if (t >= count) break;
            // top: the row's maximum less the offset
            const float z = across_sum(sum[t]) + 1e-8f * __builtin_amdgcn_exp2f(fmaxf(across_max(top[t]), -offset[t]));
            const float inv = 1.f / z;
            const int at = (from + t) * 16 + l16;
            if (at < c) {
                o_rows.store(vq[t], o[t] * inv);
                if (quad == 0) g.lse[h * g.N + T0 + at] = offset[t] + __builtin_amdgcn_logf(z);
            }
        }
    };
    Task task;
    while (work.next(g, task)) {
        const int all = (task.c + 15) >> 4;
        for (int from = task.rank * F_TILES; from < all; from += task.team * F_TILES) {
            const int count = min(F_TILES, all - from);
            if (g.word[task.T] >> 31) run(task.c, task.T, from, count, std::true_type{});
            else run(task.c, task.T, from, count, std::false_type{});
        }
    }
    __syncthreads();
    const float m = largest_of_workgroup(most, bias);           // (the table has been read)
    if (threadIdx.x == 0) g.largest_v[blockIdx.x] = m;
}

// row operands: of 16-bit tokens as they are, of fp32 tokens as pairs
template <typename T> struct Row {
    Frag<T> f;
    __device__ __forceinline__ void set(const Frag<T>& raw, const f32x4&, float) { f = raw; }
    static __device__ __forceinline__ f32x4 times(const Row& a, const Row& b, const f32x4& c) { return mma(a.f, b.f, c); }
};
template <> struct Row<float> {
    Pair x;
    __device__ __forceinline__ void set(const Frag<float>&, const f32x4& v, float by) { x = split(v * by); }
    static __device__ __forceinline__ f32x4 times(const Row& a, const Row& b, const f32x4& c) {
        return mma32(both(a.x.l, a.x.l), both(b.x.h, b.x.l), mma32(both(a.x.h, a.x.h), both(b.x.h, b.x.l), c));
    }
};

// ------------------------------------------------------------------------------------------
// backward: a wavefront holds keys and values of its tiles and walks over the window's queries, 16 at a time.  Scores, P and dS are formed once: dV = P^T dO
// and dK = scale dS^T Q stay in accumulators, dS is turned through LDS for dQ = scale dS K (the wavefronts of a window add theirs in a fixed
// order), and its entries are added to the head's table in LDS.
// ------------------------------------------------------------------------------------------
constexpr int B_RESIDENT = 2;                                            // wavefronts a SIMD
// Of a wavefront: three tiles to turn, one of which holds D of the step's queries before.  The largest table of a window of 384 positions, 2475 rows of 6 x 8 x 8, then
// leaves room for two workgroups, 81 868 bytes each (one: 111 600 tokens fp32 166 us, two 120).
constexpr int WAVE_LDS = 3 * TURN - (PITCH - 16);
// P is formed times 2^P_BITS, so that exponents lie around zero, where fp32 rounds them least, and split times 2^P_MORE on top: 22 bits of it down to 2^-28, and 2^-50
constexpr int P_BITS = 7, P_MORE = 7;
// Steps between two meetings of a window's wavefronts.  With one sum a row of the table: at every step 143 us (225 700 tokens fp16) and 130 (8100 in nearly full windows),
// every other one 142 and 126, at every fourth 141 and 124; fp32 within 2 % of each other.  Four do not fit LDS twice beside two sums of 13^3 rows.
constexpr int GROUP = 2;
enum class How { plain, masked, exact };   // windows of one mask region, of several; fp32 products of the rows as they are
template <typename T, bool TABLE> __global__ __launch_bounds__(WAVES * 64, B_RESIDENT) void flash_window_backward_kernel(Args g) {
    constexpr bool PAIRS = sizeof(T) == 4, SCALED = !std::is_same<T, __half>::value;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, l16 = lane & 15, quad = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // LDS: [2][rows] sums, [2][rows / 32] bits of rows that are +inf, -inf; tiles to turn; exchange; bias of the head
    const int words = (g.rows + 31) >> 5;
    unsigned long long* const sums = reinterpret_cast<unsigned long long*>(lds);
    uint32_t* const infinite = reinterpret_cast<uint32_t*>(sums + (TABLE ? 2 * g.rows : 0));
    float* const tiles_lds = reinterpret_cast<float*>(infinite + (TABLE ? (2 * words + 3) / 4 * 4 : 0));
    float* const turn = tiles_lds + wave * WAVE_LDS;
    float* const deltas = turn;
    float* const shared = tiles_lds + WAVES * WAVE_LDS;                  // [2][GROUP][WAVES][256]
    int* const stops = reinterpret_cast<int*>(shared + 2 * GROUP * WAVES * 256);   // [2][8]
    float* const bias = shared + 2 * GROUP * WAVES * 256 + 16;
    const uint32_t bias_at = lds_address(bias), sums_at = lds_address(sums) - 2 * bias_at;   // of a row's sum, with twice the address of its bias
    int h, first;
    place(g.H, h, first);
    Work<KT> work(g, first);
    stage_table(g, h, bias);
    if (threadIdx.x < 16) stops[threadIdx.x] = 0;
    int unit = 0, top = 0;                                               // the table's sums are in units of 2^unit, and 2^(unit - fine); |dS| < 2^top
    const int fine = g.bits - KEEPS;
    if constexpr (TABLE) {
        for (int i = threadIdx.x; i < 2 * g.rows; i += WAVES * 64) sums[i] = 0;
        for (int i = threadIdx.x; i < 2 * words; i += WAVES * 64) infinite[i] = 0;
        float mo = 0.f, mv = 0.f, o[DELTA_BLOCKS / 64], v[FORWARD_BLOCKS / 64];   // requested together
#pragma unroll
        for (int i = 0; i < DELTA_BLOCKS / 64; ++i) o[i] = g.largest[h * g.n_largest + min(i * 64 + lane, g.n_largest - 1)];
#pragma unroll
        for (int i = 0; i < FORWARD_BLOCKS / 64; ++i) {                  // of the head's workgroups, as place() deals them
            const int b = min(i * 64 + lane, g.n_largest_v - 1);
            v[i] = g.largest_v[((b >> 3) * g.H + h) * 8 + (b & 7)];
        }
#pragma unroll
        for (int i = 0; i < DELTA_BLOCKS / 64; ++i) mo = fmaxf(mo, o[i]);
#pragma unroll
        for (int i = 0; i < FORWARD_BLOCKS / 64; ++i) mv = fmaxf(mv, v[i]);
        for (int o = 1; o < 64; o <<= 1) mo = fmaxf(mo, __shfl_xor(mo, o, 64)), mv = fmaxf(mv, __shfl_xor(mv, o, 64));
        top = __builtin_amdgcn_readfirstlane(bound_of_ds(mo, mv)), unit = top - g.bits;
    }
    __syncthreads();
    const int D = g.H * HD;
    const Rows<T> q_rows(g.qkv, g.N, 3 * D, h * HD), k_rows(g.qkv, g.N, 3 * D, D + h * HD), v_rows(g.qkv, g.N, 3 * D, 2 * D + h * HD), do_rows(g.dout, g.N, D, h * HD);
    const Rows<T> dq_rows(g.dqkv, g.N, 3 * D, h * HD), dk_rows(g.dqkv, g.N, 3 * D, D + h * HD), dv_rows(g.dqkv, g.N, 3 * D, 2 * D + h * HD);
    const Buffer order = buffer(g.order, g.N), word = buffer(g.word, g.N), lses = buffer(g.lse + h * g.N, g.N), dots = buffer(g.delta, g.N * g.H);
    const float scale2 = g.scale * LOG2E, unscale = 1.f / scale2;

    // A window's tiles.  Returns -1, or, where pieces of one scale do not hold the rows, how many steps are in the table's sums: the window is then done
    // again with fp32 products (by all of a workgroup that shares windows), with the rest of the steps.
    auto run = [&](const Task& task, int added, auto how_tag) __attribute__((always_inline)) -> int {
        constexpr How HOW = decltype(how_tag)::value;
        constexpr bool EXACT = HOW == How::exact, MASK = HOW != How::plain;
        constexpr uint32_t KEPT = MASK ? 0x7fffffffu : INDEX;            // of a word
        const int c = task.c, T0 = task.T, all = (c + 15) >> 4;
        Row<T> k[KT], v[KT];
        Held<T> kt[KT];
        f32x4 dk[KT], dv[KT];
        uint32_t pk[KT];
        int vk[KT];
        bool stop = false;
        int done = 0;                                                    // steps in the table's sums
        int ek = 0, ev = 0, eq = 30, eo = 60;                            // scales
        if (task.team > 1) __syncthreads();                              // the exchange of the last window has been read
        if (c > 0) {
            Frag<T> raw_k[KT], raw_v[KT];
#pragma unroll
            for (int t = 0; t < KT; ++t) {
                dk[t] = dv[t] = f32x4{0.f, 0.f, 0.f, 0.f};
                vk[t] = load1(order, l16 * 4, (T0 + (task.first + t) * 16) * 4);   // behind the window's end: some other token
                pk[t] = load1(word, l16 * 4, (T0 + (task.first + t) * 16) * 4) & KEPT;
            }
            if constexpr (!EXACT) {
#pragma unroll
                for (int t = 0; t < KT; ++t) k_rows.row(vk[t], raw_k[t]), v_rows.row(vk[t], raw_v[t]);
                uint32_t mk[KT], mv[KT], most_k = 0, most_v = 0;
#pragma unroll
                for (int t = 0; t < KT; ++t) {
                    const bool live = t < task.tiles && (task.first + t) * 16 + l16 < c;
                    keep(live, raw_k[t]), keep(live, raw_v[t]);
                    mk[t] = over_quads(largest4(widened(raw_k[t]))), mv[t] = over_quads(largest4(widened(raw_v[t])));
                    most_k = max(most_k, mk[t]), most_v = max(most_v, mv[t]);
                }
                if (SCALED) ek = scale_for(over_rows(most_k), 30);
                ev = scale_for(over_rows(most_v), 30);
                bool lost = most_k >= NOT_FINITE || most_v >= NOT_FINITE;
#pragma unroll
                for (int t = 0; t < KT; ++t) {
                    if (SCALED) lost = lost || too_large(mk[t], ek) || too_small<T>(mk[t], ek);
                    lost = lost || too_large(mv[t], ev) || (PAIRS && too_small<T>(mv[t], ev));
                    const f32x4 kw = widened(raw_k[t]);
                    k[t].set(raw_k[t], kw, power(ek)), v[t].set(raw_v[t], widened(raw_v[t]), power(ev));
                    kt[t].set(turned(turn, SCALED ? kw * power(ek) : kw));
                }
                stop = __any(lost);
                if (task.team == 1 && stop) return 0;
            }
        }
        struct Strip {                                                   // 16 queries
            int voxel;
            Frag<T> q, d_o;
            u32x4 w;
            f32x4 lse;
            float delta;                                                 // of the lane's row
        };
        auto voxel_of = [&](int s) { return (int)load1(order, l16 * 4, (T0 + s * 16) * 4); };
        auto request = [&](int s, int voxel, Strip& x) {
            x.voxel = voxel;
            q_rows.row(voxel, x.q);
            do_rows.row(voxel, x.d_o);
            x.delta = __builtin_bit_cast(float, load1(dots, __umul24((uint32_t)voxel, (uint32_t)g.H) * 4, h * 4));
            x.w = load4(word, quad * 16, (T0 + s * 16) * 4);
            x.lse = __builtin_bit_cast(f32x4, load4(lses, quad * 16, (T0 + s * 16) * 4));
        };
        Strip ahead;
        int voxel_ahead = 0;
        if (c > 0) {
            request(0, voxel_of(0), ahead);
            if (all > 1) voxel_ahead = voxel_of(1);
        }
        const int steps = task.team > 1 ? task.steps : all;
#pragma clang loop unroll(disable)
        for (int s = 0; s < steps; ++s) {
            f32x4 dq = {0.f, 0.f, 0.f, 0.f};
            Sum dq_sum = {dq, dq};
            int voxel = 0;
            if (s < all) {
                Strip now = ahead;
                voxel = now.voxel;
                if (s + 1 < all) request(s + 1, voxel_ahead, ahead);
                if (s + 2 < all) voxel_ahead = voxel_of(s + 2);
                const int last = c - 1 - s * 16;
                float odd = 0.f;
                if (last < 15) {                                         // nothing behind the window's end
                    keep(l16 <= last, now.q), keep(l16 <= last, now.d_o);
                    if (l16 > last) now.delta = 0.f;
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (quad * 4 + j > last) now.lse[j] = INFINITY;
                        else odd += now.lse[j] * 0.f;
                } else {
                    odd = not_finite(now.lse);
                }
                const f32x4 qw = widened(now.q), ow = widened(now.d_o);
                if (quad == 0) deltas[l16] = now.delta;
                lanes_meet();
                const f32x4 delta = *reinterpret_cast<const f32x4*>(deltas + quad * 4);   // of the rows of an accumulator
                lanes_meet();
                uint32_t pq[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) pq[j] = (now.w[j] & KEPT) + (uint32_t)g.offset4 + (MASK ? 0 : bias_at);
                int es = 0;                                              // dS 2^es lies below 2^15
                if constexpr (!EXACT) {
                    const uint32_t mq = SCALED ? over_quads(largest4(qw)) : 0, mo = over_quads(largest4(ow));
                    if (__any((SCALED && too_large(mq, eq)) || too_large(mo, eo))) {
                        const int q_to = SCALED ? min(eq, scale_for(over_rows(mq), 30)) : eq, o_to = min(eo, scale_for(over_rows(mo), 60));
                        const float bk = power(max(-126, q_to - eq + o_to - eo)), bv = SCALED ? power(max(-126, o_to - eo)) : 1.f;
#pragma unroll
                        for (int t = 0; t < KT; ++t) dk[t] *= bk, dv[t] *= bv;
                        eq = q_to, eo = o_to;
                    }
                    stop = stop || __any(odd != odd || !(fabsf(now.delta) < power(32 - eo - ev)) || (SCALED && (too_large(mq, eq) || too_small<T>(mq, eq))) || too_large(mo, eo) || too_small<T>(mo, eo));
                    if (stop && task.team == 1) return s;
                    es = eo + ev - 18;
                }
                // Added to it, a value times 2^es is rounded to the unit of the sums; below `small`, to the finer one of the second sums
                const uint32_t unit_hi = (uint32_t)(0x3ff80000 + ((52 + unit + es) << 20)), fine_hi = unit_hi - ((uint32_t)fine << 20);
                const float small = power(max(-127, min(127, top - fine + es)));
                const uint32_t fine_at = sums_at + 8 * g.rows;
                auto add = [&](uint32_t at, float x) __attribute__((always_inline)) {
                    const bool low = fabsf(x) < small;
                    // (fp32: fewer registers that way, 12 spilled less, 225 700 tokens 230 -> 221 us; 16 bit: 3 % slower)
                    const uint32_t hi = PAIRS ? unit_hi - (low ? (uint32_t)fine << 20 : 0) : low ? fine_hi : unit_hi;
                    const unsigned long long b = __builtin_bit_cast(unsigned long long, (double)x + __builtin_bit_cast(double, (unsigned long long)hi << 32));
                    const unsigned long long n = (unsigned long long)((uint32_t)(b >> 32) - hi) << 32 | (uint32_t)b;
                    __hip_atomic_fetch_add((LdsLong*)(uintptr_t)(2 * at + (PAIRS ? sums_at + (low ? 8 * g.rows : 0) : low ? fine_at : sums_at)), n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                };
                if constexpr (!EXACT) {
                  if (!stop) {
                    const float cq = SCALED ? power(eq) : 1.f, co = SCALED ? power(eo) : 1.f;
                    Row<T> q, d_o;
                    q.set(now.q, qw, cq), d_o.set(now.d_o, ow, co);
                    Column<T> qt, dot;
                    qt.set(turned(turn + 2 * TURN, SCALED ? qw * cq : qw));
                    dot.set(turned(turn + 2 * TURN, SCALED ? ow * co : ow));
                    const float by_s = PAIRS ? power(eq + ek) : 1.f, by_p = PAIRS ? power(eo + ev) : 1.f, to_s = PAIRS ? scale2 * power(-eq - ek) : scale2,
                                to_ds = PAIRS ? power(-18 - P_BITS) : power(es - P_BITS);
                    const f32x4 a0 = (now.lse - (float)P_BITS) * (-unscale * by_s), d0 = delta * -by_p;  // what the accumulators start from: P comes out times 2^P_BITS
                    auto tiles = [&](auto from_tag, auto count_tag) __attribute__((always_inline)) {
                        constexpr int FROM = decltype(from_tag)::value, COUNT = decltype(count_tag)::value;
                        f32x4 p[COUNT], ds[COUNT];
                        uint32_t at[COUNT][4];
#pragma unroll
                        for (int i = 0; i < COUNT; ++i) {
                            const int t = FROM + i;
                            const f32x4 acc = Row<T>::times(q, k[t], a0), dp = Row<T>::times(d_o, v[t], d0);
#pragma unroll
                            for (int j = 0; j < 4; ++j) {
                                const uint32_t d = pq[j] - pk[t];
                                at[i][j] = MASK ? (d & INDEX) + bias_at : d;
                                float x = fmaf(acc[j], to_s, lds_float(at[i][j]));
                                if (MASK && d >> 15) x += MASKED;
                                p[i][j] = __builtin_amdgcn_exp2f(fminf(x, P_BITS + 0.5f));   // (P of keys behind the window's end has no bound)
                                ds[i][j] = p[i][j] * to_ds * dp[j];
                            }
                        }
                        if constexpr (TABLE) {
#pragma unroll
                            for (int i = 0; i < COUNT; ++i)
                                if (FROM + i < task.tiles && (task.first + FROM + i) * 16 + l16 < c) {
#pragma unroll
                                    for (int j = 0; j < 4; ++j) add(at[i][j], ds[i][j]);
                                }
                        }
#pragma unroll
                        for (int i = 0; i < COUNT; ++i) {
                            const int t = FROM + i;
                            const f32x4 dst = turned(turn + i * TURN, ds[i]);
                            dv[t] = dot.times(split_fine<P_MORE>(p[i]), dv[t]);
                            dk[t] = qt.times(split_fine(ds[i]), dk[t]);
                            kt[t].add(split_fine(dst), dq_sum);
                        }
                    };
                    // An odd last tile by itself where a tile is bound by what it issues: backward with the table's gradient, windows of 7^3, 112 700 tokens fp32 111 -> 106 us,
                    // 225 700 214 -> 203.  16-bit tokens wait more than they issue, and a second form of the loop's body costs them 2 % (225 700 fp16 145 and 149).
                    auto two = [&](auto from_tag) __attribute__((always_inline)) {
                        const int more = task.tiles - decltype(from_tag)::value;
                        if (more > 1 || (!PAIRS && more > 0)) tiles(from_tag, std::integral_constant<int, 2>{});
                        else if (more > 0) tiles(from_tag, std::integral_constant<int, 1>{});
                    };
                    two(std::integral_constant<int, 0>{});
                    two(std::integral_constant<int, 2>{});
                    two(std::integral_constant<int, 4>{});
#pragma unroll
                    for (int j = 0; j < 4; ++j) dq[j] = __builtin_amdgcn_ldexpf(dq_sum.total()[j], -es - ek);
                    ++done;
                  }
                } else {
                    const Frag<float> qt = {turned(turn + 2 * TURN, qw)}, dot = {turned(turn + 2 * TURN, ow)};
                    const f32x4 a0 = now.lse * -unscale, d0 = -delta;
                    const float most = top > 126 ? 3.0e38f : power(max(-126, top));
#pragma unroll
                    for (int t = 0; t < KT; ++t) {
                        if (t >= task.tiles) break;
                        const bool live = (task.first + t) * 16 + l16 < c;
                        Frag<T> raw_k, raw_v;
                        k_rows.row(vk[t], raw_k), v_rows.row(vk[t], raw_v);
                        keep(live, raw_k), keep(live, raw_v);
                        const f32x4 acc = mma(now.q, raw_k, a0), dp = mma(now.d_o, raw_v, d0);
                        Frag<float> pf, df;
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            const bool taken = live && quad * 4 + j <= last;
                            const uint32_t d = pq[j] - pk[t], at = (d & INDEX) + bias_at;
                            float x = fmaf(acc[j], scale2, lds_float(at));
                            if (d >> 15) x += MASKED;
                            pf.v[j] = taken ? __builtin_amdgcn_exp2f(x) : 0.f;
                            df.v[j] = taken ? pf.v[j] * dp[j] : 0.f;
                            if (TABLE && taken && s >= added) {
                                if (fabsf(df.v[j]) <= most) add(at, df.v[j]);
                                else {
                                    const uint32_t row = (d & INDEX) >> 2, bit = 1u << (row & 31);
                                    if (!(df.v[j] < 0.f)) atomicOr(infinite + (row >> 5), bit);
                                    if (!(df.v[j] > 0.f)) atomicOr(infinite + words + (row >> 5), bit);
                                }
                            }
                        }
                        const Frag<float> ktf = {turned(turn, widened(raw_k))}, dst = {turned(turn + TURN, df.v)};
                        dv[t] = mma(dot, pf, dv[t]);
                        dk[t] = mma(qt, df, dk[t]);
                        dq = mma(ktf, dst, dq);
                    }
                }
            }
            if (task.team == 1) {
                if (s * 16 + l16 < c) dq_rows.store(voxel, dq * g.scale);
                continue;
            }
            // The wavefronts of a window meet every GROUP steps and add the parts of the steps between, each those of its own steps: the same order on every run.
            // Parts are not written again before the next meeting but one.
            float* const parts = shared + (s / GROUP & 1) * GROUP * WAVES * 256;
            if (s < all) *reinterpret_cast<f32x4*>(parts + (s % GROUP * WAVES + wave) * 256 + lane * 4) = dq;
            if (s % GROUP != GROUP - 1 && s != steps - 1) continue;
            int voxels[GROUP];
#pragma unroll
            for (int i = 0; i < GROUP; ++i) voxels[i] = voxel_of(s / GROUP * GROUP + i);
            int* const stopped = stops + (s / GROUP & 1) * 8;
            if (!EXACT && lane == 0) stopped[wave] = stop;
            __syncthreads();
            if constexpr (!EXACT) {
                bool any = false;
#pragma unroll
                for (int w = 0; w < WAVES; ++w) any = any || stopped[w];
                if (__builtin_amdgcn_readfirstlane(any)) return done;
            }
#pragma unroll
            for (int i = 0; i < GROUP; ++i) {
                const int step = s / GROUP * GROUP + i;
                if (step > s || (step & (task.team - 1)) != task.rank || step * 16 + l16 >= c) continue;
                f32x4 sum = {0.f, 0.f, 0.f, 0.f};
                for (int w = 0; w < task.team; ++w) sum += *reinterpret_cast<const f32x4*>(parts + (i * WAVES + wave - task.rank + w) * 256 + lane * 4);
                dq_rows.store(voxels[i], sum * g.scale);
            }
        }
        const int sk = EXACT ? 0 : -(eo + ev - 18) - (SCALED ? eq : 0), sv = EXACT ? 0 : -P_BITS - P_MORE - (SCALED ? eo : 0);
#pragma unroll
        for (int t = 0; t < KT; ++t)
            if (t < task.tiles && (task.first + t) * 16 + l16 < c) {
                f32x4 x, y;
#pragma unroll
                for (int j = 0; j < 4; ++j) x[j] = __builtin_amdgcn_ldexpf(dk[t][j] * g.scale, sk), y[j] = __builtin_amdgcn_ldexpf(dv[t][j], sv);
                dk_rows.store(vk[t], x);
                dv_rows.store(vk[t], y);
            }
        return -1;
    };
    Task task;
    while (work.next(g, task)) {
        const bool several = task.c > 0 && g.word[task.T] >> 31;
        const int added = several ? run(task, 0, std::integral_constant<How, How::masked>{}) : run(task, 0, std::integral_constant<How, How::plain>{});
        if (added >= 0) run(task, added, std::integral_constant<How, How::exact>{});
    }
    if constexpr (TABLE) {
        __syncthreads();
        float* const to = g.partial + ((int64_t)h * g.per_head + first) * g.rows;
        for (int i = threadIdx.x; i < g.rows; i += WAVES * 64) {
            float sum = (float)(ldexp((double)(long long)sums[i], unit) + ldexp((double)(long long)sums[g.rows + i], unit - fine));
            const bool up = infinite[i >> 5] >> (i & 31) & 1, down = infinite[words + (i >> 5)] >> (i & 31) & 1;
            if (up) sum = down ? __builtin_nanf("") : INFINITY;
            else if (down) sum = -INFINITY;
            to[i] = sum;
        }
    }
}

// d table[row][h]: a workgroup adds 16 rows of a head, 64 threads a row, in a fixed order
__global__ __launch_bounds__(1024) void flash_window_table_kernel(const float* __restrict__ partial, int per_head, int rows, int H, float* __restrict__ d_table) {
    __shared__ double part[64][17];
    const int r = threadIdx.x & 15, q = threadIdx.x >> 4, h = blockIdx.y, row = blockIdx.x * 16 + r;
    double s = 0.;
    if (row < rows) {
        const float* const src = partial + (int64_t)h * per_head * rows + row;
        for (int i = q; i < per_head; i += 64) s += src[(int64_t)i * rows];
    }
    part[q][r] = s;
    __syncthreads();
    if (q == 0 && row < rows) {
        double total = 0.;
        for (int k = 0; k < 64; ++k) total += part[k][r];
        d_table[(int64_t)row * H + h] = (float)total;
    }
}

static int add_table(const float* partial, int per_head, int rows, int H, float* d_table, hipStream_t s) {
    hipLaunchKernelGGL(flash_window_table_kernel, dim3((unsigned)((rows + 15) / 16), (unsigned)H), dim3(1024), 0, s, partial, per_head, rows, H, d_table);
    return launch_ok("flash_window_backward, table");
}

static size_t backward_lds(int rows, bool table) {
    const int words = (rows + 31) / 32;
    return (table ? (size_t)rows * 16 + (2 * words + 3) / 4 * 16 : 0) + (size_t)(WAVES * WAVE_LDS + 2 * GROUP * WAVES * 256 + 16 + rows) * sizeof(float);
}

template <typename T, bool TABLE> static int launch_backward(Args g, hipStream_t s) {
    const size_t lds = backward_lds(g.rows, TABLE);
    if (lds > 64 * 1024)
        SSWIN_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(flash_window_backward_kernel<T, TABLE>), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    hipLaunchKernelGGL((flash_window_backward_kernel<T, TABLE>), dim3((unsigned)(g.per_head * g.H)), dim3(WAVES * 64), lds, s, g);
    return launch_ok("flash_window_backward");
}

template <typename T> static int run_forward(const Args& g, hipStream_t s) {
    hipLaunchKernelGGL(flash_window_forward_kernel<T>, dim3((unsigned)(g.per_head * g.H)), dim3(WAVES * 64), (size_t)(WAVES * TURN + g.rows) * sizeof(float), s, g);
    return launch_ok("flash_window_forward");
}

template <typename T> static int run_backward(Args g, float* delta, float* largest, float* d_table, hipStream_t s) {
    const int64_t parts = g.N * g.H * (HD / 4);
    // at least the lanes of one voxel
    const int blocks = (int)std::max<int64_t>((g.H * (HD / 4) + 255) / 256, std::min<int64_t>(DELTA_BLOCKS, (parts + 1023) / 1024));
    hipLaunchKernelGGL((flash_window_delta_kernel<T>), dim3(blocks), dim3(256), 0, s, static_cast<const T*>(g.dout), static_cast<const T*>(g.out), parts, g.H, delta,
                       largest);
    if (int rc = launch_ok("flash_window_backward, delta")) return rc;
    g.delta = delta, g.largest = largest, g.n_largest = blocks;
    // what a workgroup adds to a row of the table: at most one value a query, MOST tiles of them a round
    const int64_t rounds = (g.windows + g.per_head - 1) / g.per_head, most = std::min<int64_t>(g.N, rounds * MOST * 16);
    g.bits = std::min(50, __builtin_clzll((unsigned long long)most) - 2);
    if (!d_table) return launch_backward<T, false>(g, s);
    if (int rc = launch_backward<T, true>(g, s)) return rc;
    return add_table(g.partial, g.per_head, g.rows, g.H, d_table, s);
}

}  // namespace window
}  // namespace flash
}  // namespace sswin

using namespace sswin;
using namespace sswin::flash;
using namespace sswin::flash::window;

// Where most windows are a workgroup's, no more workgroups than the same number of rounds takes: the others would only share its SIMD (8100 tokens in 50
// nearly full windows, 24 heads: 40 workgroups a head 71.7 us, 32 67)
static int forward_per_head(int dtype, int64_t N, int windows, int H) {
    const int m = per_head(windows, H, forward_resident(dtype == SSWIN_F32 ? 4 : 2)), rounds = (windows + m - 1) / m;
    return N <= (int64_t)windows * 2 * F_TILES * 16 ? m : ((windows + rounds - 1) / rounds + 7) / 8 * 8;
}

static int window_args(const char* what, int dtype, const int32_t* plan, int64_t g_cap, int64_t groups, const int32_t* tokens, const int32_t* word,
                       const int32_t* list, int64_t N, int H, int hd, int n, const void* qkv, float scale, const float* table, int rows, int offset0, void* out,
                       float* lse, Args& g) {
    SSWIN_CHECK(H > 0 && groups > 0 && groups <= g_cap && groups % H == 0 && offset0 >= 0 && sswin_flash_window_list_ints(dtype, N, H, hd, n, rows, groups / H),
                "%s: not a shape it takes", what);
    SSWIN_CHECK(plan && tokens && word && list && qkv && table && out && lse, "%s: null pointer", what);
    SSWIN_CHECK(((uintptr_t)qkv | (uintptr_t)out) % 16 == 0, "%s: pointers must be 16-byte aligned", what);
    g.plan = plan, g.g_cap = g_cap, g.order = tokens, g.word = reinterpret_cast<const uint32_t*>(word), g.list = list, g.N = N, g.windows = (int)(groups / H);
    g.largest_v = reinterpret_cast<float*>(const_cast<int32_t*>(list)) + LIST_HEAD + g.windows, g.n_largest_v = forward_per_head(dtype, N, g.windows, H);
    g.H = H, g.rows = rows, g.offset4 = offset0 * 4, g.scale = scale, g.table = table, g.qkv = qkv, g.out = out, g.lse = lse;
    return 0;
}

extern "C" {

// A window costs these kernels a tile of 16 rows and a wavefront's start however few tokens it has; flash_attention.hip packs small windows into 32 rows, and pays by
// the token and, more than these, by the pair.  Lines through 110 000 tokens in windows of 12, 24 and 60 (fp32, 3 heads: forward and backward 34 us longer here, 11 and 64
// shorter) are as 1000 windows, 29 tokens, 1.1 pairs: windows of one size c cross at c = 20.  There both take the same within 12 % but where launches are what takes the
// time (0.75): windows of 3^3, 5^3, 7^3, all types, 3 to 12 heads, 30 000 to 220 000 tokens; at 12 these take 0.9 to 1.35 times as long, at 6 1.15 to 2.1, at 2 2.4 to 4.5; at
// 24 0.78 to 0.99, at 60 0.63 to 0.85.  Few large windows among small ones are these kernels' (200 of 200 tokens, 3800 of 3: 330 -> 211 us), which the tokens of the mean
// window, 13, would not tell.
int sswin_flash_window_faster(int64_t N, int64_t windows, int64_t pairs) { return 1000 * windows <= 30 * N + pairs; }

size_t sswin_flash_window_list_ints(int dtype, int64_t N, int H, int hd, int n, int rows, int64_t windows) {
    return hd == HD && n <= MOST * 16 && H <= MOST_HEADS && windows > 0 && windows <= LIST_WINDOWS && sswin_flash_supported(dtype, N, H, hd, rows) && N * 3 * H * hd < 1ll << 30
               ? (size_t)LIST_HEAD + windows + FORWARD_BLOCKS : 0;
}

int sswin_flash_window_tokens(const int32_t* plan, int64_t g_cap, int64_t groups, const int32_t* tokens, int64_t N, int H, int n, const int32_t* code,
                              const int8_t* mask, int nmw, int32_t* word, int32_t* list, void* stream) {
    SSWIN_CHECK(N > 0 && N < MAX_TOKENS && n > 0 && n <= MOST * 16 && H > 0 && groups > 0 && groups <= g_cap && groups % H == 0 && groups / H <= LIST_WINDOWS,
                "flash_window_tokens: bad sizes");
    SSWIN_CHECK(plan && tokens && code && word && list && (!mask || nmw > 0), "flash_window_tokens: null pointer");
    const int windows = (int)(groups / H), per = LIST_THREADS / 64;
    hipLaunchKernelGGL(flash_window_tokens_kernel, dim3((unsigned)(1 + (windows + per - 1) / per)), dim3(LIST_THREADS), 0, static_cast<hipStream_t>(stream), plan,
                       g_cap, windows, H, tokens + 3 * N, code, mask, nmw, n, reinterpret_cast<uint32_t*>(word), list);
    return launch_ok("flash_window_tokens");
}

int sswin_flash_window_forward(int dtype, const int32_t* plan, int64_t g_cap, int64_t groups, const int32_t* tokens, const int32_t* word, int32_t* list,
                               int64_t N, int H, int hd, int n, const void* qkv, float scale, const float* table, int rows, int offset0, void* out, float* lse,
                               void* stream) {
    Args g = {};
    if (int rc = window_args("flash_window_forward", dtype, plan, g_cap, groups, tokens, word, list, N, H, hd, n, qkv, scale, table, rows, offset0, out, lse, g))
        return rc;
    g.per_head = forward_per_head(dtype, N, g.windows, H);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == SSWIN_F32) return run_forward<float>(g, s);
    if (dtype == SSWIN_F16) return run_forward<__half>(g, s);
    return run_forward<__hip_bfloat16>(g, s);
}

size_t sswin_flash_window_backward_workspace_bytes(int64_t N, int H, int rows, int64_t windows) {
    Carver c(nullptr, 0);
    c.take<float>((size_t)H * N);
    c.take<float>((size_t)DELTA_BLOCKS * H);
    c.take<float>((size_t)per_head((int)windows, H, B_RESIDENT) * H * rows);
    return c.used;
}

int sswin_flash_window_backward(int dtype, const int32_t* plan, int64_t g_cap, int64_t groups, const int32_t* tokens, const int32_t* word, const int32_t* list,
                                int64_t N, int H, int hd, int n, const void* qkv, float scale, const float* table, int rows, int offset0, const void* out,
                                const float* lse, const void* dout, void* dqkv, float* d_table, void* ws, size_t ws_bytes, void* stream) {
    Args g = {};
    if (int rc = window_args("flash_window_backward", dtype, plan, g_cap, groups, tokens, word, list, N, H, hd, n, qkv, scale, table, rows, offset0,
                             const_cast<void*>(out), const_cast<float*>(lse), g))
        return rc;
    SSWIN_CHECK(dout && dqkv && ws && ((uintptr_t)dout | (uintptr_t)dqkv) % 16 == 0, "flash_window_backward: gradients at 16 bytes and a workspace");
    Carver c(ws, ws_bytes);
    float* const delta = c.take<float>((size_t)H * N);
    float* const largest = c.take<float>((size_t)DELTA_BLOCKS * H);
    g.per_head = per_head(g.windows, H, B_RESIDENT);
    g.partial = c.take<float>((size_t)g.per_head * H * rows);
    SSWIN_CHECK(c.ok(), "flash_window_backward: workspace of %zu bytes, %zu are needed", ws_bytes, c.used);
    g.dout = dout, g.dqkv = dqkv;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == SSWIN_F32) return run_backward<float>(g, delta, largest, d_table, s);
    if (dtype == SSWIN_F16) return run_backward<__half>(g, delta, largest, d_table, s);
    return run_backward<__hip_bfloat16>(g, delta, largest, d_table, s);
}

}  // extern "C"
