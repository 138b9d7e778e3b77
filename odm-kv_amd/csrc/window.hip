// Observation-window attention mass: p[h,t] = mean over the W window queries and the G query heads of a
// kv-head of softmax_t(q . k_t * scaling), causal inside the window, over the core tokens t >= n_sink.
//
// This is the per-query form of the scorer's attention estimate (the reference scores with ONE query per
// head, the mean query: kvquant/scorer.py:285-318; here every query of the last W positions votes).  It is a
// true dense contraction, [G W, 128] x [128, T] per kv-head, and runs on the 16-bit matrix instructions
// (v_mfma_f32_32x32x16_f16 / _bf16) with exact products of the model's own 16-bit values and fp32 sums.
//
// Two passes over K, the logits are never stored:
//   pass 1  rows of the matrix product = tokens, columns = queries: a lane owns a query and keeps that
//           query's running statistics over the tokens it sees; per-workgroup results go to `stats`
//   stats   merge per query -> M + log2 Z
//   pass 2  rows = queries, columns = tokens: a lane owns a token and sums exp2(s - M - log2 Z) over the queries
// The same two operand fragments serve both passes; only their roles (A or B) swap.
// A workgroup keeps 128 tokens in LDS, the next 128 on their way into its other half (global_load_lds: no registers, no wait until they are
// needed), and each of its eight wavefronts holds 32 queries in registers and goes over all of the tokens: a query's statistics then stay in two
// registers of a lane, and what a query brings along (its weight, its position) is fetched once.
// What bounds it: 67 MB of keys a pass (12 us at the rate these reads reach, the first tile of 64 KB a compute unit 5 to 9 us after the start) and
// 13 us of products and vector work (67 million exponentials at half the vector rate, a subtraction and an addition each), of which a tile's part
// runs under the next tile's way.  32k tokens of 8 heads, 64 queries, bf16, us a pass: 41.5 + 33.8 -> 29.3 + 28.1; whole calls of 32
// heads over 8, us: 600 tokens 32 -> 18, 8k 40.7 -> 27.1, 32k 75 -> 61, 131k 234 -> 183 (fp16 239 -> 188).  Before, 64 tokens lay in a
// wavefront's registers and 256 queries in LDS: all keys were asked for before the first product, every wavefront closed 256 queries' statistics
// for its 64 tokens, and the tokens inside the window divided by W at every logit, in wavefronts that ran 10 us longer than the others.
// Tried, no faster: 16 wavefronts and four tiles under way (33 + 29), 256 tokens in one tile (33.5 + 28.7), wave priorities, the next products
// issued ahead of a block's vector work.
#include <algorithm>
#include "common.h"

#define WIN_WAVES 8
#define WIN_THREADS (WIN_WAVES * 64)
#define WIN_TILE 128         // tokens of a workgroup at a time, in LDS
#define WIN_TILE_BYTES (WIN_TILE * HD * 2)
#define WIN_LDS (2 * WIN_TILE_BYTES + 2 * WIN_WAVES * WIN_TILE * 4)

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct WinArgs {
    const void* K;
    const void* Q;        // [Hq, W, 128], same 16-bit type as K; the queries of kv-head h are rows h G W .. (h+1) G W
    int64_t sH, sT;
    int Hkv, G, W, R, T, Tc, n_sink, tile, tiles, nchunks, qpos0;     // tokens of a tile (WIN_TILE, or 2 WIN_TILE and a single tile), tiles of a workgroup
    int qblocks, slots;   // blocks of 32 queries of a kv-head; of them at a time in a workgroup (1, 2, 4 or 8: its wavefronts share the tokens out 8 / slots ways)
    float inv_w;          // 1 / W
    float c;              // scaling * log2(e): logits in base-2 units
    float* stats;         // [Hkv][nchunks * 8 / slots][R][2]
    float* mz;            // [Hkv R]: maximum + log2(sum), both in base-2 units
    float* p;             // [Hkv][Tc]
    float* kn2;           // [Hkv][Tc]: |k|^2, or null (pass 1 holds every key anyway)
};

template <int DT>
__device__ static inline f32x16 win_mfma(uint4 a, uint4 b, f32x16 c) {
    if constexpr (DT == ODMKV_F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// merge two (max, sum) pairs kept in base-2 units (a maximum of -inf: nothing seen yet, the sum is 0, or NaN where a logit was; either stays
// so times exp2(-inf).  A branch for it kept the statistics kernel from asking for eight entries at once: 0.9 us a call)
__device__ static inline void ms2_merge(float& m, float& s, float m2, float s2) {
    const float mn = fmaxf(m, m2), by = mn > -INFINITY ? mn : 0.0f;
    s = s * __builtin_amdgcn_exp2f(m - by) + s2 * __builtin_amdgcn_exp2f(m2 - by);
    m = mn;
}

// index (0..31) inside a 32-row block of accumulator register r of a lane in wave half `half`
__device__ static inline int acc_row(int r, int half) { return 8 * (r >> 2) + 4 * half + (r & 3); }

// the other half of the wave's value of v (lane ^ 32)
__device__ static inline float other_half(float v, int half) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(half ? r[0] : r[1]);
}

template <int DT>
__device__ static inline float squares8(const uint4& k) {
    const uint32_t w[4] = {k.x, k.y, k.z, k.w};
    float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float x0 = Elem<DT>::to_f32((uint16_t)(w[e] & 0xffffu)), x1 = Elem<DT>::to_f32((uint16_t)(w[e] >> 16));
        s0 = __fmaf_rn(x0, x0, s0);
        s1 = __fmaf_rn(x1, x1, s1);
    }
    return s0 + s1;
}

// A query's statistics over the tokens that a lane has seen: the sum of exp2(s - ref).  The reference point is the largest s or up to 4 below it (an
// exponent of that size is still rounded to 2^-22): sixteen tokens whose sum is at most 16 need no maximum, which most have not but the first.
// A logit that is NaN makes the sum NaN, wherever it comes, and the query then votes for nothing.
struct QueryStat { float ref, sum; };
#define WIN_RISE 16.0f

// sixteen raw products, c of each in base-2 units, join the statistics
__device__ static inline void fold_products(const f32x16& p, float c, QueryStat& q) {
    float z0 = 0.0f, z1 = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; r += 2) {
        z0 += __builtin_amdgcn_exp2f(__fmaf_rn(p[r], c, -q.ref));
        z1 += __builtin_amdgcn_exp2f(__fmaf_rn(p[r + 1], c, -q.ref));
    }
    float z = z0 + z1;
    if (__any(!(z <= WIN_RISE))) {                                  // (with a reference point of -inf z is infinite or NaN)
        float ref = q.ref;
#pragma unroll
        for (int r = 0; r < 16; ++r) ref = fmaxf(ref, p[r] * c);
        z = 0.0f;
        const float by = ref > -INFINITY ? ref : 0.0f;              // (nothing but -inf and NaN: sums to 0 or NaN)
#pragma unroll
        for (int r = 0; r < 16; ++r) z += __builtin_amdgcn_exp2f(__fmaf_rn(p[r], c, -by));
        q.sum *= __builtin_amdgcn_exp2f(q.ref - by);
        q.ref = ref;
    }
    q.sum += z;
}
// the same where some of them are not to be seen (-inf, all in base-2 units already)
__device__ static inline void fold_masked(const f32x16& s, QueryStat& q) {
    float ref = q.ref;
#pragma unroll
    for (int r = 0; r < 16; ++r) ref = fmaxf(ref, s[r]);
    const float by = ref > -INFINITY ? ref : 0.0f;
    float z = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) z += __builtin_amdgcn_exp2f(s[r] - by);
    q.sum = __fmaf_rn(q.sum, __builtin_amdgcn_exp2f(q.ref - by), z);
    q.ref = ref;
}

// a tile of keys on its way from memory into LDS without passing through registers: 16 bytes a lane, a wavefront's 1024 bytes one behind the other from `to` on
__device__ static inline void request_to_lds(const uint16_t* from, uint32_t to) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(from), "{m0}"(to) : "memory");      // (m0 is the place in LDS)
}

template <int DT, int PASS>
__global__ __launch_bounds__(WIN_THREADS, 4) void window_kernel(WinArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];                 // two tiles of [WIN_TILE][256 bytes] or one of twice as many rows, then part
    float* part = reinterpret_cast<float*>(smem + 2 * WIN_TILE_BYTES);        // pass 2: [2][WIN_WAVES][WIN_TILE] or [WIN_WAVES][2 WIN_TILE]
    // heads vary fastest: a die of the chip (workgroups go round over the eight) then keeps few heads' queries in its L2
    const int h = blockIdx.x % a.Hkv, chunk = blockIdx.x / a.Hkv, tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);      // (scalar: what follows from it branches, it does not mask lanes)
    const int lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int chunk_t0 = chunk * a.tiles * a.tile, tiles = min(a.tiles, (a.Tc - chunk_t0 + a.tile - 1) / a.tile);
    const int slot = wave & (a.slots - 1), share = wave / a.slots, shares = WIN_WAVES / a.slots;
    // Operand fragments: the matrix instruction contracts over 16 elements per step, 8 from either half of the wave, elements 16 st + 8 half .. + 7.
    uint4 q[8];                                                     // the queries of a block: row 32 qb + col
    float ml[PASS == 2 ? 16 : 1];                                   // M + log2 Z: exp2(s - ml) = exp2(s - M) / Z
    const auto request_queries = [&](int qb) {
        int c = col, hf = half;                                     // opaque: the addresses are worked out here, not carried round the loops
        asm volatile("" : "+v"(c), "+v"(hf));
        const int row = 32 * qb + c;
        const uint16_t* src = reinterpret_cast<const uint16_t*>(a.Q) + ((size_t)h * a.R + row) * HD + 8 * hf;
#pragma unroll
        for (int st = 0; st < 8; ++st) q[st] = row < a.R ? *reinterpret_cast<const uint4*>(src + 16 * st) : make_uint4(0u, 0u, 0u, 0u);
        if (PASS == 2) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {                          // rows without a query take weight 0: exp2(0 - inf)
                const int row = 32 * qb + acc_row(r, hf);
                const float v = a.mz[h * a.R + min(row, a.R - 1)];
                ml[r] = row < a.R ? v : INFINITY;
            }
        }
    };
    // Piece p (16 bytes) of row r of a tile lies at piece p ^ (r % 16) of the row's place: the reads of consecutive rows fall on distinct banks.
    // Rows past the end repeat the last one and are masked.
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) uint8_t*)smem;
    const auto request_tile = [&](int i) {
        const uint16_t* base = reinterpret_cast<const uint16_t*>(a.K) + (size_t)h * a.sH + (size_t)a.n_sink * a.sT;
        const auto rows_of = [&](int half_tile) {
#pragma unroll
            for (int k = 0; k < WIN_TILE * 16 / WIN_THREADS; ++k) {
                const int e = tid + WIN_THREADS * k, row = e >> 4, piece = (e & 15) ^ (row & 15);
                const int t = min(chunk_t0 + i * a.tile + half_tile * WIN_TILE + row, a.Tc - 1);
                request_to_lds(base + (size_t)t * a.sT + 8 * piece, lds0 + ((i & 1) + half_tile) * WIN_TILE_BYTES + (WIN_THREADS * k + 64 * wave) * 16);
            }
        };
        rows_of(0);
        if (a.tile > WIN_TILE) rows_of(1);
    };
    // Loads return in the order of their requests: the queries, out of the L2, before the keys, out of memory.
    if (slot < a.qblocks) request_queries(slot);
    request_tile(0);
    QueryStat stat = {-INFINITY, 0.0f};
    const int row_start = col * 256 + ((half ^ (col & 15)) << 4);
#pragma unroll 1
    for (int i = 0; i <= tiles; ++i) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");      // this tile has come, and every wavefront is done with the one before
        const int t0 = chunk_t0 + i * a.tile;
        if (i + 1 < tiles) request_tile(i + 1);                     // (under way while this one is computed)
        if (PASS == 2 && i > 0 && tid < a.tile && t0 - a.tile + tid < a.Tc) {
            // the last tile's votes: of the wavefronts that took this token's block, in their order
            const float* from = part + ((i & 1) ^ 1) * WIN_WAVES * WIN_TILE + ((tid >> 5) & (shares - 1)) * a.slots * a.tile + tid;
            float p = 0.0f;
            for (int w = 0; w < min(a.slots, a.qblocks); ++w) p += from[w * a.tile];
            a.p[(size_t)h * a.Tc + t0 - a.tile + tid] = p / (float)a.R;
        }
        if (i == tiles) break;
        const uint8_t* tile = smem + (i & 1) * WIN_TILE_BYTES;
        const int n_tok = min(a.tile, a.Tc - t0), blocks = (n_tok + 31) >> 5;       // of 32 tokens
        // keys at or before every window query need no causal test, and only the last block of all ends past the tokens
        const int plain = min(max(a.qpos0 + 1 - a.n_sink - t0, 0), n_tok) >> 5;
        if (PASS == 1 && a.kn2 != nullptr && wave < blocks) {
            float s = 0.0f;
#pragma unroll
            for (int st = 0; st < 8; ++st) s += squares8<DT>(*reinterpret_cast<const uint4*>(tile + 32 * 256 * wave + (row_start ^ (st << 5))));
            s += other_half(s, half);
            if (half == 0 && 32 * wave + col < n_tok) a.kn2[(size_t)h * a.Tc + t0 + 32 * wave + col] = s;
        }
#pragma unroll 1
        for (int qb = slot; qb < a.qblocks; qb += a.slots) {        // (more than one: a single tile a workgroup)
            if (qb != slot) {
                request_queries(qb);
                stat = {-INFINITY, 0.0f};
            }
            const auto products = [&](int tb, int row_start) {
                f32x16 acc;
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
                for (int st = 0; st < 8; ++st) {
                    const uint4 k = *reinterpret_cast<const uint4*>(tile + 32 * 256 * tb + (row_start ^ (st << 5)));
                    acc = PASS == 1 ? win_mfma<DT>(k, q[st], acc) : win_mfma<DT>(q[st], k, acc);
                }
                return acc;
            };
            // a row's place in the window, row % W: the quotient is at least 1 / (2 W), 2^-13, from a whole number, its error below G 2^-22
            const auto place = [&](int row) { return row - (int)(((float)row + 0.5f) * a.inv_w) * a.W; };
            const auto vote = [&](int tb, float p) {                // pass 2: a token's votes of this block of queries
                p += other_half(p, half);
                float* at = part + (i & 1) * WIN_WAVES * WIN_TILE + wave * a.tile + 32 * tb + col;
                if (half == 0) *at = qb == slot ? p : *at + p;
            };
            int tb = share;
#pragma unroll 1
            for (; tb < plain; tb += shares) {
                const f32x16 s = products(tb, row_start);
                if constexpr (PASS == 1) fold_products(s, a.c, stat);
                else {
                    float p[2] = {0.0f, 0.0f};
#pragma unroll
                    for (int r = 0; r < 16; ++r) p[r & 1] += __builtin_amdgcn_exp2f(__fmaf_rn(s[r], a.c, -ml[r]));
                    vote(tb, p[0] + p[1]);
                }
            }
#pragma unroll 1
            for (; tb < blocks; tb += shares) {
                int at = row_start;                                  // opaque, as in request_queries
                asm volatile("" : "+v"(at));
                f32x16 s = products(tb, at);
                if constexpr (PASS == 1) {
                    // this lane's query: its position decides which of the last keys it sees
                    const int last = min(a.qpos0 + place(32 * qb + col) - a.n_sink, a.Tc - 1) - t0 - 32 * tb - 4 * half;
#pragma unroll
                    for (int r = 0; r < 16; ++r) s[r] = acc_row(r, 0) <= last ? s[r] * a.c : -INFINITY;
                    fold_masked(s, stat);
                } else {
                    const int pos = a.n_sink + t0 + 32 * tb + col - a.qpos0;         // this lane's token, seen by the window's queries from there on
                    float p = 0.0f;
                    int first = 32 * qb + 4 * half;                  // opaque: sixteen rows' places worked out ahead of the loop take as many registers
                    asm volatile("" : "+v"(first));
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float e = __builtin_amdgcn_exp2f(__fmaf_rn(s[r], a.c, -ml[r]));
                        p += pos > place(first + acc_row(r, 0)) ? 0.0f : e;
                    }
                    vote(tb, p);
                }
            }
            if (PASS == 1 && i + 1 == tiles) {
                // the other half of the wave holds the same query's other tokens
                ms2_merge(stat.ref, stat.sum, other_half(stat.ref, half), other_half(stat.sum, half));
                const int row = 32 * qb + col;
                if (half == 0 && row < a.R)
                    reinterpret_cast<float2*>(a.stats)[((size_t)h * a.nchunks * shares + chunk * shares + share) * a.R + row] = make_float2(stat.ref, stat.sum);
            }
        }
    }
}

// merge a query's statistics, one of every share of a workgroup's tokens, into M + log2 Z: 64 queries a workgroup, a lane each, the entries shared out over its wavefronts
#define WIN_STAT_WAVES 16
__global__ __launch_bounds__(WIN_STAT_WAVES * 64) void window_stats_kernel(WinArgs a) {
    __shared__ float ms[WIN_STAT_WAVES][64], ss[WIN_STAT_WAVES][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = blockIdx.y;
    const int row = blockIdx.x * 64 + lane, n = a.nchunks * (WIN_WAVES / a.slots);
    const float2* st = reinterpret_cast<const float2*>(a.stats) + (size_t)h * n * a.R + min(row, a.R - 1);
    float m = -INFINITY, s = 0.0f;
    for (int e0 = wave; e0 < n; e0 += 8 * WIN_STAT_WAVES) {         // eight entries under way
        float2 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = e0 + i * WIN_STAT_WAVES;
            v[i] = e < n ? st[(size_t)e * a.R] : make_float2(-INFINITY, 0.0f);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) ms2_merge(m, s, v[i].x, v[i].y);
    }
    ms[wave][lane] = m; ss[wave][lane] = s;
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 1; w < WIN_STAT_WAVES; ++w) ms2_merge(m, s, ms[w][lane], ss[w][lane]);
    // a query that sees no key at all (cannot happen when the window lies behind the sinks) votes for nothing
    if (row < a.R) a.mz[(size_t)h * a.R + row] = (m > -INFINITY && s > 0.0f) ? m + __builtin_amdgcn_logf(s) : INFINITY;
}

// blocks of 32 queries that a workgroup's wavefronts take at a time
static inline int win_slots(int R) { return R > 128 ? 8 : R > 64 ? 4 : R > 32 ? 2 : 1; }

// Tiles of a workgroup: as many as two workgroups a compute unit take in one round.  Where the queries are more than its wavefronts hold, they come
// again for every tile: a single one, of twice as many tokens from three a compute unit on (28 heads over 4, us with 128 and 256 tokens: 8k tokens
// 26.8 / 34.7, 20k 51.0 / 53.8, 32k 64.8 / 58.8, 131k 217 / 178; before 59, 64, 68 and 195).
static inline bool win_turns(int R) { return R > 32 * WIN_WAVES; }
static inline int64_t win_all_tiles(int Hkv, int Tc) { return (int64_t)Hkv * ((Tc + WIN_TILE - 1) / WIN_TILE); }
static inline int win_tile(int Hkv, int R, int Tc, int cus) { return win_turns(R) && win_all_tiles(Hkv, Tc) > 3 * cus ? 2 * WIN_TILE : WIN_TILE; }
static inline int win_tiles(int Hkv, int R, int Tc, int cus) {
    return win_turns(R) ? 1 : (int)std::max<int64_t>(1, (win_all_tiles(Hkv, Tc) + 2 * cus - 1) / (2 * cus));
}
static inline int win_chunks(int tile, int tiles, int Tc) { return (Tc + tiles * tile - 1) / (tiles * tile); }

extern "C" size_t odmkv_window_attention_workspace_bytes(int Hkv, int Hq, int W, int T) {
    if (Hkv <= 0 || Hq <= 0 || W <= 0 || T <= 0) return 0;
    const size_t rows = (size_t)Hq * W;                   // (the chunks of single small tiles: no call has more)
    return align_up(rows * (size_t)win_chunks(WIN_TILE, 1, T) * (WIN_WAVES / win_slots(Hq / Hkv * W)) * 8, 256) + align_up(rows * 8, 256);
}

template <int DT>
static int run_window(const WinArgs& a, hipStream_t st) {
    ODMKV_ALLOW_LDS((window_kernel<DT, 1>), WIN_LDS);
    ODMKV_ALLOW_LDS((window_kernel<DT, 2>), WIN_LDS);
    const dim3 grid((unsigned)a.nchunks * a.Hkv), block(WIN_THREADS);
    hipLaunchKernelGGL((window_kernel<DT, 1>), grid, block, WIN_LDS, st, a);
    ODMKV_CHECK_LAUNCH("window_kernel<1>");
    hipLaunchKernelGGL(window_stats_kernel, dim3((a.R + 63) / 64, a.Hkv), dim3(WIN_STAT_WAVES * 64), 0, st, a);
    ODMKV_CHECK_LAUNCH("window_stats_kernel");
    hipLaunchKernelGGL((window_kernel<DT, 2>), grid, block, WIN_LDS, st, a);
    ODMKV_CHECK_LAUNCH("window_kernel<2>");
    return 0;
}

static int window_attention(const void* K, int dtype, int Hkv, int T, int64_t stride_h, int64_t stride_t,
                            const void* Q, int Hq, int W, int q_pos0, int n_sink, float scaling,
                            float* p, float* kn2, void* workspace, size_t workspace_bytes, void* stream) {
    ODMKV_CHECK_ARG(K && Q && p && workspace, "window_attention: null pointer");
    ODMKV_CHECK_ARG(dtype == ODMKV_F16 || dtype == ODMKV_BF16,
                    "window_attention: keys and queries must be float16 or bfloat16 (dtype %d)", dtype);
    ODMKV_CHECK_ARG(Hkv > 0 && Hq > 0 && Hq % Hkv == 0, "window_attention: bad head counts Hkv=%d Hq=%d", Hkv, Hq);
    ODMKV_CHECK_ARG(W >= 1 && W <= 4096, "window_attention: bad window %d", W);
    ODMKV_CHECK_ARG(n_sink >= 0 && T > n_sink, "window_attention: need T > n_sink (T=%d, n_sink=%d)", T, n_sink);
    ODMKV_CHECK_ARG(q_pos0 >= n_sink, "window_attention: the window must lie behind the sinks (q_pos0=%d, n_sink=%d)", q_pos0, n_sink);
    ODMKV_CHECK_ARG(stride_h % 8 == 0 && stride_t % 8 == 0 && stride_t >= HD, "window_attention: strides must keep rows 16-byte aligned");
    ODMKV_CHECK_ARG(((uintptr_t)K & 15) == 0 && ((uintptr_t)Q & 15) == 0, "window_attention: K and Q must be 16-byte aligned");
    ODMKV_CHECK_ARG(workspace_bytes >= odmkv_window_attention_workspace_bytes(Hkv, Hq, W, T), "window_attention: workspace too small");
    WinArgs a;
    a.K = K; a.Q = Q; a.sH = stride_h; a.sT = stride_t;
    a.Hkv = Hkv; a.G = Hq / Hkv; a.W = W; a.R = a.G * W; a.T = T; a.Tc = T - n_sink; a.n_sink = n_sink;
    const int cus = compute_units();
    a.tile = win_tile(Hkv, a.R, a.Tc, cus); a.tiles = win_tiles(Hkv, a.R, a.Tc, cus); a.nchunks = win_chunks(a.tile, a.tiles, a.Tc); a.qpos0 = q_pos0;
    a.qblocks = (a.R + 31) / 32; a.slots = win_slots(a.R);
    a.inv_w = 1.0f / (float)W;
    a.c = scaling * 1.4426950408889634f;
    const size_t rows = (size_t)Hq * W;
    a.stats = (float*)workspace;                          // the workspace is sized for the chunks of all T tokens
    a.mz = (float*)((char*)workspace + align_up(rows * (size_t)win_chunks(WIN_TILE, 1, T) * (WIN_WAVES / a.slots) * 8, 256));
    a.p = p; a.kn2 = kn2;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == ODMKV_F16) return run_window<ODMKV_F16>(a, st);
    return run_window<ODMKV_BF16>(a, st);
}

extern "C" int odmkv_window_attention(const void* K, int dtype, int Hkv, int T, int64_t stride_h, int64_t stride_t,
                                      const void* Q, int Hq, int W, int q_pos0, int n_sink, float scaling,
                                      float* p, void* workspace, size_t workspace_bytes, void* stream) {
    return window_attention(K, dtype, Hkv, T, stride_h, stride_t, Q, Hq, W, q_pos0, n_sink, scaling, p, nullptr, workspace, workspace_bytes, stream);
}

// The same, and |k|^2 of the core tokens, which the first pass holds all keys for: the risk score is spared a pass of its own over
// them (12 us of 165 for 32k tokens of 8 heads).
extern "C" int odmkv_window_attention_norms(const void* K, int dtype, int Hkv, int T, int64_t stride_h, int64_t stride_t,
                                            const void* Q, int Hq, int W, int q_pos0, int n_sink, float scaling,
                                            float* p, float* kn2, void* workspace, size_t workspace_bytes, void* stream) {
    ODMKV_CHECK_ARG(kn2, "window_attention: null pointer");
    return window_attention(K, dtype, Hkv, T, stride_h, stride_t, Q, Hq, W, q_pos0, n_sink, scaling, p, kn2, workspace, workspace_bytes, stream);
}
