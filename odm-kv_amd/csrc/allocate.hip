// Lagrangian bit allocation: for every non-sink token pick  argmin_k  s * eps_k + lambda * b_k,
// with lambda found by bisection so that the mean of the chosen widths meets the row's budget,
// then close the remaining gap by moving the lowest- (or highest-) scored tokens one level.
//
// The search is the fixed sequence the host formulation runs: lambda = 1, up to 8 widenings of the
// bracket (x10 each), 64 halvings, one final assignment.  Each of its 74 steps asks one question: is the mean at
// this lambda above the budget?  Far from the answer the question needs no pass over the scores.  A window [la, lb]
// of multipliers is kept such that the mean is above the budget at every lambda <= la and within it at every
// lambda >= lb, by more than the rounding of any cost could change; the launches narrow it, and the last of them replays
// the sequence, answering what lies outside the window from the window and the rest by an exact sum over the
// few tokens whose level is not the same all over it:
//   range     the least and the largest positive score;
//   scan      a histogram between them, a thousand bins of equal steps of the bit pattern;
//   search    (one workgroup a row) a guess from the bins: where the budget's multiplier must lie by the bins' edges, and where
//             it lies if the scores are spread evenly in a bin.  Nothing rests on it but the time;
//   narrow    one pass over the scores at eight multipliers, the guess' ends and three pairs closing in on its middle: the window;
//   collect   how many tokens take which level wherever in the window lambda lies, and the list of the others;
//   finish    (one workgroup a row) the replay over that list: the multiplier, the histogram of levels, the gap;
//   assign    levels out, and the candidates for the repair's moves;
//   repair    (one workgroup a row) the moves.
// What was 24 launches, ten of which walked all scores with fifteen multipliers each, is eight, and eight multipliers once.
// us a call: 4096 scores 107 -> 53, 2 rows of 12432 107 -> 55, 4 of 262144 158 -> 69, one of 1048576 183 -> 80.
// Every workgroup writes its partial sums with plain stores and is done (the scan's alone add to the row's histogram by atomics).  The next launch begins,
// in every workgroup, by adding up the row's partial sums of the launch before (a few hundred
// numbers); the row's first workgroup also writes the new state down for the launch after.  Nothing waits on another workgroup
// and the host is never consulted.  All sums are integers, so the result does not depend on the order
// in which workgroups run. 
//
// Arithmetic is kept exactly as the host formulation it replaces: fp32 products rounded
// separately and then added (no fused multiply-add), lambda rounded to fp32 before use, the
// first (lowest-width) level wins a tie, avg = fp32(sum) / fp32(n), bracket and gap in fp64.
//
// What the window rests on.  A cost s * eps_k + lambda * b_k is linear in (s, lambda), so the difference of two levels' costs is
// least at a corner of any box of scores and multipliers.  Computed costs are off by less than 2^-22 of their size (the sum of two
// products, errors not negative); where one level beats another by 2^-20 and 1e-36 (products in the subnormal range) at all
// corners it therefore beats it, as computed, throughout the box.  And a level with fewer bits that loses by
// that much at some lambda loses at every smaller one (its difference falls with lambda), one with more bits at every larger
// one: a sum that is above the budget with every token that is nearly tied counted at its least is above it for all smaller
// multipliers.  A cost with a negative error is a difference of two products, whose sizes add up to no more than the cost and twice the
// negative one: there the margin grows by 2^-18 of the score times the largest negative error, which is linear in (s, lambda) as well
// (eight of the roundings above, 3 x 2^-24, each side, and two where the second best is below zero).  Infinite errors are constant in lambda (and 0 * inf, a NaN, meets
// zero scores alone, which take the first level in any case); NaN, and -inf behind another, are given the infinity that every token
// treats alike (odmkv_allocate).  Without a window for such tables the replay asked all tokens, in one workgroup a row.
// Us a call, one row of 262144: with a negative error 3900 -> 62, an infinite one 3900 -> 59, eviction at an infinite cost 2640 -> 61.
#include <algorithm>
#include <cmath>
#include "common.h"

#define NLV ODMKV_MAX_LEVELS
#define N_HALVE 64
#define NGRID 8                               // multipliers of a narrowing pass
#define SLOTS 16                              // partial sums per workgroup: NGRID sums and how far near ties may move them, or NLV levels and the list's length
#define EV_THREADS 512
#define EV_TPT 2                              // tokens per thread of the assignment
#define EV_TOKENS (EV_THREADS * EV_TPT)
#define EV_WGS 512ll                          // workgroups a pass is cut for over all rows
#define EV_BIG 2                              // tokens per thread and run of a call with more than 256 x EV_THREADS of them
#define EV_MAX_CHUNKS 256                     // workgroups of a row in a pass
#define CAND_MAX 16                           // repair moves of at most this many tokens take the short path
#define HB_BINS 1024                          // bin 0: zeros; the last: infinities and NaN; between them equal steps of the bit pattern
#define MAX_TURN 2048                         // rows of a turn: what the histograms' workspace is cut for
#define LAMBDA_CAP 100000008.0f               // the fp32 number behind the largest multiplier that is asked for, 1e8
#define LAMBDA_LEAST 0x1p-66f                 // no multiplier that is asked for or returned is less: 64 halvings of 1 and the middle of what is left
#define KEEP (1.0f - 0x1p-20f)                // one cost beats another by more than rounding: other * KEEP > best + slack()
#define TINY 1e-36f

struct RowState {
    double target, gap, lam;
    float la, lb;            // the window: the mean is above the budget at lambda <= la, within it at lambda >= lb
    float wa, wb;            // [la, lb] above LAMBDA_LEAST, stretched to any final multiplier outside it: what "open" is decided over
    float grid[NGRID];       // the narrowing pass' multipliers, ascending
    int n_active;
    unsigned int max_finite; // bit pattern
    int has_finite, has_nonfinite;
    int final_hist[NLV];
};

struct AllocArgs {
    const float* scores;
    const uint8_t* sink_mask;
    int rows, n, period, n_sink, sink_bits, K;
    int n_chunks, iters;           // workgroups of a row in a pass, and how many runs of tokens each of them walks
    int chunk_tokens;
    int n_cand;                    // workgroups of a row in the assignment
    int n_scan;                    // workgroups of a row in the range and the histogram
    // the levels on the lower hull of (bits, error): beyond a ratio score / lambda of step_at[i] a token takes step_bits[i] more than before
    int n_steps, first_bits;
    float step_at[NLV], step_bits[NLV];
    float slack_s;                 // 2^-18 of the largest negative error's size
    float eps[NLV];
    float bitsf[NLV];
    int nominal[NLV];
    const double* target;          // device, [rows]
    uint2* range;                  // [rows, n_scan]: bit patterns of the least positive and the largest finite score
    unsigned int* hist;            // [rows, HB_BINS]
    unsigned int* partial;         // [2][rows, n_chunks, SLOTS]: the narrowing pass', the collecting one's
    float* open;                   // [rows, n]: the open tokens' scores, a region per chunk
    uint8_t* open_n;               // [rows, n]: how many tokens an entry stands for
    unsigned long long* cand;      // [rows, n_cand, NLV, CAND_MAX]: per move of the repair
    RowState* state;               // [2][rows]: the search and the finish leave half 1, the collecting pass half 0
    int32_t* bits_out;
    int32_t* level_counts;
    double* lambda_out;
};

__device__ static inline bool is_sink(const AllocArgs& a, int row, int i) {
    if (a.sink_mask) return a.sink_mask[(size_t)row * a.n + i] != 0;
    return a.n_sink > 0 && (i % a.period) < a.n_sink;
}

// what a cost of a token must be beaten by, beside the factor KEEP
__device__ static inline float slack(const AllocArgs& a, float s) { return __fmaf_rn(s, a.slack_s, TINY); }

// torch's clamp(min=0) / non-finite patch / nan_to_num, in that order
__device__ static inline float clean_score(float v, bool patch, float top) {
    if (!(v != v)) v = fmaxf(v, 0.0f);                // clamp(min=0) keeps NaN
    if (patch && !isfinite(v)) v = top;
    if (v != v) v = 0.0f;
    else if (v == INFINITY) v = 3.4028234663852886e38f;
    return v;
}

struct Cleaner {
    bool patch;
    float top;
    __device__ inline Cleaner(const RowState& st) : patch(st.has_finite && st.has_nonfinite), top(__uint_as_float(st.max_finite)) {}
    __device__ inline float operator()(float v) const { return clean_score(v, patch, top); }
};

__device__ static inline int wave_sum_int(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
    return v;
}

// the same on the vector ALU alone: shifts within the rows of 16 lanes, then the rows' sums handed on; all lanes get the sum
__device__ static inline int wave_sum_dpp(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);      // row_shr 1, 2, 4, 8: lane 15 of a row holds the row
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);      // row_bcast 15 into rows 1 and 3, row_bcast 31 into rows 2 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return __builtin_amdgcn_readlane(v, 63);
}

// ---- the range of a row's scores, and a histogram over it ----
#define SC_THREADS 512
#define SC_BIG 16                             // scores per thread of a call with more than 256 workgroups of SC_SMALL a thread
#define SC_SMALL 4
#define SC_MAX 256                            // workgroups a row: 128 of the large, 256 of the small at most
// bit pattern of a score as the allocation sees it, 0x7f800000 and above for one that is not finite
__device__ static inline unsigned int score_bits(float v) { return v != v ? 0x7fffffffu : __float_as_uint(fmaxf(v, 0.0f)) & 0x7fffffffu; }

template <int TPT>
__device__ static inline void scan_load(const AllocArgs& a, int row, unsigned int (&b)[TPT], bool (&on)[TPT]) {
    float raw[TPT];
    const int i0 = blockIdx.x * (SC_THREADS * TPT) + threadIdx.x;
    int at = a.n_sink > 0 ? i0 % a.period : 0;               // place in the period, carried along: a division per score took longer than reading it
    const int step = a.n_sink > 0 ? SC_THREADS % a.period : 0;
#pragma unroll
    for (int e = 0; e < TPT; ++e) {                          // all reads first: one round trip, not TPT
        const int i = i0 + e * SC_THREADS;
        on[e] = i < a.n && !(a.sink_mask ? a.sink_mask[(size_t)row * a.n + i] != 0 : at < a.n_sink);
        raw[e] = on[e] ? a.scores[(size_t)row * a.n + i] : 0.0f;
        at += step;
        at -= at >= a.period ? a.period : 0;
    }
#pragma unroll
    for (int e = 0; e < TPT; ++e) b[e] = score_bits(raw[e]);
}

template <int TPT>
__global__ __launch_bounds__(SC_THREADS) void alloc_range_kernel(AllocArgs a) {
    __shared__ unsigned int least[SC_THREADS / 64], most[SC_THREADS / 64];
    const int row = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (blockIdx.x == 0 && a.level_counts && tid < a.K) a.level_counts[row * a.K + tid] = 0;
    if (blockIdx.x == 0 && tid < HB_BINS / 4) reinterpret_cast<uint4*>(a.hist + (size_t)row * HB_BINS)[tid] = make_uint4(0u, 0u, 0u, 0u);
    unsigned int b[TPT];
    bool on[TPT];
    scan_load<TPT>(a, row, b, on);
    unsigned int lo = 0x7f800000u, hi = 0u;
#pragma unroll
    for (int e = 0; e < TPT; ++e) {
        const bool finite = on[e] && b[e] < 0x7f800000u;
        if (finite && b[e] != 0u) lo = min(lo, b[e]);
        if (finite) hi = max(hi, b[e]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, (unsigned int)__shfl_xor((int)lo, o, WAVE));
        hi = max(hi, (unsigned int)__shfl_xor((int)hi, o, WAVE));
    }
    if (lane == 0) { least[wave] = lo; most[wave] = hi; }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < SC_THREADS / 64; ++w) { lo = min(lo, least[w]); hi = max(hi, most[w]); }
        a.range[(size_t)row * a.n_scan + blockIdx.x] = make_uint2(lo, hi);
    }
}

// bins 1 .. HB_BINS - 2: (bits - base) >> shift
struct Bins { unsigned int base, top; int shift; };
__device__ static inline Bins row_bins(const AllocArgs& a, int row) {       // every wavefront by itself
    const int lane = threadIdx.x & 63;
    unsigned int lo = 0x7f800000u, hi = 0u;
#pragma unroll
    for (int u = 0; u < SC_MAX / 64; ++u) {
        if (lane + 64 * u < a.n_scan) {
            const uint2 r = a.range[(size_t)row * a.n_scan + lane + 64 * u];
            lo = min(lo, r.x); hi = max(hi, r.y);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo = min(lo, (unsigned int)__shfl_xor((int)lo, o, WAVE));
        hi = max(hi, (unsigned int)__shfl_xor((int)hi, o, WAVE));
    }
    Bins r;
    r.top = hi;
    r.base = lo < hi ? lo : hi;
    const unsigned int range = hi - r.base;
    r.shift = max(0, 32 - __clz((int)range) - 10);           // (1024 = 2^10 steps at most; one more shift below if two are too many)
    if ((range >> r.shift) > (unsigned int)(HB_BINS - 3)) ++r.shift;
    return r;
}

template <int TPT>
__global__ __launch_bounds__(SC_THREADS) void alloc_scan_kernel(AllocArgs a) {
    __shared__ unsigned int h[HB_BINS];
    const int row = blockIdx.y, tid = threadIdx.x;
    unsigned int b[TPT];
    bool on[TPT];
    scan_load<TPT>(a, row, b, on);
    const Bins bins = row_bins(a, row);
    for (int i = tid; i < HB_BINS; i += SC_THREADS) h[i] = 0u;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < TPT; ++e)
        if (on[e]) atomicAdd(&h[b[e] == 0u ? 0u : b[e] >= 0x7f800000u ? (unsigned int)HB_BINS - 1u : 1u + ((b[e] - bins.base) >> bins.shift)], 1u);
    __syncthreads();
    unsigned int* out = a.hist + (size_t)row * HB_BINS;
    for (int i = tid; i < HB_BINS; i += SC_THREADS)
        if (h[i]) atomicAdd(&out[i], h[i]);
}

// the window after the mean's bounds at one multiplier (sums of widths over the row, with nearly tied tokens at their least / largest)
__device__ static inline void shrink(RowState& st, float lambda, float least, float most) {
    const float nf = (float)st.n_active;
    if ((double)(least / nf) > st.target) st.la = fmaxf(st.la, lambda);
    if (!((double)(most / nf) > st.target)) st.lb = fminf(st.lb, lambda);
}

// ---- a guess from the histogram ----
// A token's level depends on score / lambda alone, so a row's sum at any lambda is a count of the scores beyond lambda times the
// hull's few ratios: one look per ratio into the running counts.  A thread takes a multiplier of its own: all 95 octaves in 1023
// steps, then the stretch between the last that is surely above and the first that is surely within the budget in 1023 more, twice.
#define SE_THREADS 1024
#define SE_LEAST 0x1p-68f                     // below every multiplier that is asked for
__global__ __launch_bounds__(SE_THREADS) void alloc_search_kernel(AllocArgs a) {
    __shared__ unsigned int from[HB_BINS + 1];               // scores in this bin and above
    __shared__ unsigned int wave_tot[SE_THREADS / 64];
    __shared__ int last_above, first_within, last_over;
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    static_assert(HB_BINS == SE_THREADS, "a bin per thread");
    unsigned int mine = a.hist[(size_t)row * HB_BINS + tid];
    const unsigned int zeros = a.hist[(size_t)row * HB_BINS], odd = a.hist[(size_t)row * HB_BINS + HB_BINS - 1];
    double target = a.target[row];                           // clamp the budget into the level range
    const Bins bins = row_bins(a, row);
    const bool has_finite = bins.top != 0u || zeros != 0u;
    if (has_finite) {                                        // infinities and NaN are taken for the largest finite score
        if (tid == HB_BINS - 1) mine = 0u;
        if (tid == (bins.top == 0u ? 0 : 1 + (int)((bins.top - bins.base) >> bins.shift))) mine += odd;
    }
    unsigned int incl = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned int up = __shfl_up(incl, o, WAVE);
        if (lane >= o) incl += up;
    }
    if (lane == 63) wave_tot[wave] = incl;
    if (tid == 0) { last_above = -1; first_within = SE_THREADS; last_over = -1; }
    __syncthreads();
    unsigned int before = incl - mine, total = 0u;
#pragma unroll
    for (int w = 0; w < SE_THREADS / 64; ++w) {
        if (w < wave) before += wave_tot[w];
        total += wave_tot[w];
    }
    from[tid] = total - before;
    if (tid == 0) from[HB_BINS] = 0u;
    __syncthreads();
    target = fmin(target, (double)a.nominal[a.K - 1]);
    target = fmax(target, (double)a.nominal[0]);
    const float budget = (float)(target * (double)total);
    // (Without a finite score, those that are not count as beyond everything.)
    float l0 = SE_LEAST, l1 = LAMBDA_CAP, guess = 1.0f;
    if (total != 0u) {
#pragma unroll 1
        for (int round = 0; round < 3; ++round) {
            const float span = log2f(l1 / l0) * (1.0f / (float)(SE_THREADS - 1)), base = l0;
            const float lambda = base * exp2f(span * (float)tid);
            float least = (float)a.first_bits * (float)total, most = least, even = least;
            for (int i = 0; i < a.n_steps; ++i) {
                const float x = lambda * a.step_at[i];
                const unsigned int xb = __float_as_uint(x);
                const unsigned int b = xb < bins.base ? 0u : min(1u + ((xb - bins.base) >> bins.shift), (unsigned int)HB_BINS - 2u);
                const unsigned int b0 = bins.base + ((b - 1u) << bins.shift);
                const float e0 = __uint_as_float(b0), e1 = __uint_as_float(b0 + (1u << bins.shift));
                const float above = (float)from[b + 1], in = b == 0u ? 0.0f : (float)from[b] - above;
                least += above * a.step_bits[i];
                most += (above + in) * a.step_bits[i];
                even += (above + in * fminf(fmaxf((e1 - x) / (e1 - e0), 0.0f), 1.0f)) * a.step_bits[i];
            }
            const unsigned long long m0 = __ballot(least > budget), m1 = __ballot(most <= budget), m2 = __ballot(even > budget);
            if (lane == 0) {
                if (m0) atomicMax(&last_above, tid + 63 - __clzll((long long)m0));
                if (m1) atomicMin(&first_within, tid + __ffsll((long long)m1) - 1);
                if (m2) atomicMax(&last_over, tid + 63 - __clzll((long long)m2));
            }
            __syncthreads();
            const int i0 = max(last_above, 0), i1 = min(first_within, SE_THREADS - 1), im = max(last_over, 0);
            __syncthreads();
            if (tid == 0) { last_above = -1; first_within = SE_THREADS; last_over = -1; }
            l0 = base * exp2f(span * (float)i0);
            l1 = base * exp2f(span * (float)i1);
            guess = base * exp2f(span * ((float)im + 0.5f));
            if (!(l1 > l0 * (1.0f + 0x1p-20f))) { l0 *= 1.0f - 0x1p-20f; l1 = fmaxf(l1, l0) * (1.0f + 0x1p-20f); }
            __syncthreads();
        }
    }
    if (tid == 0) {
        RowState& st = a.state[(size_t)a.rows + row];
        st.target = target; st.gap = 0.0; st.lam = 1.0;
        st.la = 0.0f; st.lb = LAMBDA_CAP;                    // nothing is known yet
        // the ends a little outside the bins' bounds, and three pairs around the guess: as far off as a bin is wide, an eighth and a 64th of it
        // (and no closer than where nearly every token is nearly tied)
        const float w = fmaxf(ldexpf(1.0f, bins.shift - 23), 0x1p-14f), w1 = fmaxf(w * 0x1p-3f, 0x1p-16f), w2 = fmaxf(w * 0x1p-6f, 0x1p-18f);
        const float lo = fmaxf(l0 * (1.0f - 0x1p-12f), SE_LEAST), hi = fminf(l1 * (1.0f + 0x1p-12f), 1e8f);
        const float at[NGRID] = {lo, guess * (1.0f - w), guess * (1.0f - w1), guess * (1.0f - w2),
                                 guess * (1.0f + w2), guess * (1.0f + w1), guess * (1.0f + w), hi};
        for (int i = 0; i < NGRID; ++i) st.grid[i] = fminf(fmaxf(at[i], lo), hi);
        st.n_active = (int)total;
        st.has_finite = has_finite;
        st.has_nonfinite = odd != 0u;
        st.max_finite = bins.top;
        for (int k = 0; k < NLV; ++k) st.final_hist[k] = 0;
    }
}

// The host formulation's sequence; above(lambda) answers whether the row's mean is above the budget there, and says no for every lambda
// >= lb.  (One place that asks: the finish's answer is a kilobyte of code.)
template <typename F>
__device__ static inline double replay(float lb, F above) {
    double lo = 0.0, hi = 1.0, at = 1.0;
    bool widening = true;
    for (int done = 0; done < N_HALVE;) {
        const bool over = above((float)at);
        if (widening) {
            widening = over && hi < 1e8;
            if (widening) hi *= 10.0;
        } else {
            if (over) lo = at; else hi = at;
            ++done;
        }
        if (!widening && lo == 0.0) {
            // on the way down a halving is a smaller exponent: those that end at or beyond lb are taken at once
            const int k = min(ilogb(hi) - ilogb((double)lb) - 1, N_HALVE - 1 - done);
            if (k > 0) { hi = ldexp(hi, -k); done += k; }
        }
        at = widening ? hi : (lo + hi) * 0.5;
    }
    return (lo + hi) * 0.5;
}

// Start of a pass: the state before it in `cur` (shared memory) for the whole workgroup.  The collecting pass narrows the window by what the
// narrowing one found, and the row's first workgroup writes the new state to half 0.  Ends with a barrier.
template <bool COLLECT>
__device__ static void carry_state(const AllocArgs& a, int row, RowState* cur, unsigned int* tot) {
    const int tid = threadIdx.x;
    // everything the launch needs of the last one is asked for at once: a thread's partial sums and the whole state
    unsigned int v0[8];                                      // (256 workgroups a row at most: 8 x 512)
    const int n_part = COLLECT ? a.n_chunks * SLOTS : 0;
    const unsigned int* p = a.partial + (size_t)row * a.n_chunks * SLOTS;
#pragma unroll
    for (int u = 0; u < 8; ++u) v0[u] = tid + u * EV_THREADS < n_part ? p[tid + u * EV_THREADS] : 0u;
    if (tid == 0) *cur = a.state[(size_t)a.rows + row];
    if (tid < SLOTS) tot[tid] = 0u;
    __syncthreads();
    if constexpr (COLLECT) {
        // thread tid holds slot tid % SLOTS of chunk tid / SLOTS (the block size is a multiple of SLOTS, so every
        // further element of the thread is the same slot); the four chunks of a wavefront are added across its
        // 16-lane rows before one lane per slot updates the total
        static_assert(SLOTS == 16 && EV_THREADS % SLOTS == 0, "a slot per lane of a 16-lane row");
        static_assert(EV_MAX_CHUNKS * SLOTS <= 8 * EV_THREADS, "all of a row's partial sums are under way at once");
        unsigned int v = 0u;
#pragma unroll
        for (int u = 0; u < 8; ++u) v += v0[u];
        v += (unsigned int)__shfl_xor((int)v, 16, WAVE);
        v += (unsigned int)__shfl_xor((int)v, 32, WAVE);
        if ((tid & 63) < SLOTS && v) atomicAdd(&tot[tid & (SLOTS - 1)], v);
        __syncthreads();
        if (tid == 0) {
            if (cur->n_active != 0) {
                for (int i = 0; i < NGRID; ++i) {            // sums up to 2^24: exact in fp32
                    const float sum = (float)tot[i], off = (float)tot[NGRID + i];
                    shrink(*cur, cur->grid[i], fmaxf(sum - off, 0.0f), sum + off);
                }
            }
            const float la = cur->la, lb = cur->lb;
            cur->wa = fmaxf(la, LAMBDA_LEAST); cur->wb = lb; // (at 0 itself scores whose products are all below TINY would stay open)
            // After 27 halvings behind the first that moved the lower end the bracket is narrower than the gap of two fp32 numbers, and
            // the final multiplier lies in the window.  With fewer of them, or where no bracket reaches a mean within the budget, it
            // may lie beside it: between the two that the sequence ends at if the mean inside the window is above the budget
            // everywhere, or nowhere.
            if (!(la >= 0x1p-36f && la < 1e8f)) {
#pragma unroll 1
                for (int side = 0; side < 2; ++side) {
                    const float lam = (float)replay(lb, [&](float l) { return side ? l < lb : l <= la; });
                    cur->wa = fminf(cur->wa, lam); cur->wb = fmaxf(cur->wb, lam);
                }
            }
        }
        __syncthreads();
        if (tid == 0 && blockIdx.x == 0) a.state[row] = *cur;
    }
}

// A pass over a row's scores: the sums at eight multipliers, or the settled tokens' levels and the list of
// the open ones.  A token is settled if it takes the same level at both ends (of the eight, of the window) by more than rounding could move it;
// it then takes that level throughout and is counted once.  The others are closed up in LDS and walked by eight lanes, one per multiplier.
// Every workgroup begins by adding up what the last launch's workgroups of the row left, so their number is what a
// long row pays for: a workgroup walks `iters` runs of TPT tokens per thread (at most 256 workgroups a row; short rows keep
// one token per thread).
template <int K, int TPT, bool COLLECT>
__global__ __launch_bounds__(EV_THREADS) void alloc_pass_kernel(AllocArgs a) {
    constexpr int RUN = EV_THREADS * TPT, LIST = 2 * RUN;
    __shared__ unsigned int lsum[SLOTS];
    __shared__ unsigned int tot[SLOTS];
    __shared__ RowState cur;
    __shared__ float open[COLLECT ? 1 : LIST];
    __shared__ int n_open;
    const int row = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    // the first scores are asked for first: they do not depend on the state, which takes a round trip of its own
    const int first = blockIdx.x * a.chunk_tokens, iters = min(a.iters, (a.n - first + RUN - 1) / RUN);
    float raw[TPT];
    bool active[TPT];
    auto request = [&](int it) {
#pragma unroll
        for (int e = 0; e < TPT; ++e) {
            const int i = first + it * RUN + e * EV_THREADS + tid;
            active[e] = i < a.n && !is_sink(a, row, i);
            raw[e] = active[e] ? a.scores[(size_t)row * a.n + i] : 0.0f;
        }
    };
    request(0);
    if (tid < SLOTS) lsum[tid] = 0u;
    if (tid == 0) n_open = 0;
    carry_state<COLLECT>(a, row, &cur, tot);
    const RowState& st = cur;
    if (st.n_active == 0) return;                            // (the finish looks at no partial sum of such a row)
    const Cleaner clean(st);
    float end[2][K], lb[K];                                  // fl32(lambda * b_k) at the window's ends, and at the lane's multiplier
    const int c = tid & (NGRID - 1), group = tid / NGRID;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        end[0][k] = __fmul_rn(COLLECT ? st.wa : st.grid[0], a.bitsf[k]);
        end[1][k] = __fmul_rn(COLLECT ? st.wb : st.grid[NGRID - 1], a.bitsf[k]);
        lb[k] = __fmul_rn(st.grid[c], a.bitsf[k]);
    }
    unsigned int sum = 0u, ties = 0u;
    int cnt[K];
#pragma unroll
    for (int k = 0; k < K; ++k) cnt[k] = 0;
    auto evaluate = [&](int count) {
#pragma unroll 2
        for (int i = group; i < count; i += EV_THREADS / NGRID) {
            const float s = open[i];
            float best = __fadd_rn(__fmul_rn(s, a.eps[0]), lb[0]), second = INFINITY;
            int bn = a.nominal[0];
#pragma unroll
            for (int k = 1; k < K; ++k) {
                const float cst = __fadd_rn(__fmul_rn(s, a.eps[k]), lb[k]);
                second = __builtin_amdgcn_fmed3f(cst, best, second);
                if (cst < best) { best = cst; bn = a.nominal[k]; }
            }
            sum += (unsigned int)bn;
            const float margin = best + slack(a, s);
            if (!(second * KEEP > margin)) {                 // nearly tied: by how much the level may be another at this multiplier's neighbours
                int lo = bn, hi = bn;
#pragma unroll 1
                for (int k = 0; k < K; ++k)
                    if (__fadd_rn(__fmul_rn(s, a.eps[k]), __fmul_rn(st.grid[c], a.bitsf[k])) * KEEP <= margin) { lo = min(lo, a.nominal[k]); hi = max(hi, a.nominal[k]); }
                ties += (unsigned int)max(bn - lo, hi - bn);
            }
        }
    };
    float* list = a.open + (size_t)row * a.n + first;
    uint8_t* list_n = a.open_n + (size_t)row * a.n + first;
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int e = 0; e < TPT; ++e) {
            const float s = active[e] ? clean(raw[e]) : 0.0f;
            int at[2];
            bool settled = true;
            float se[K];
#pragma unroll
            for (int k = 0; k < K; ++k) se[k] = __fmul_rn(s, a.eps[k]);
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                float best = __fadd_rn(se[0], end[side][0]), second = INFINITY;
                int bn = 0;
#pragma unroll
                for (int k = 1; k < K; ++k) {
                    const float cst = __fadd_rn(se[k], end[side][k]);
                    second = __builtin_amdgcn_fmed3f(cst, best, second);
                    if (cst < best) { best = cst; bn = k; }
                }
                at[side] = bn;
                settled = settled && second * KEEP > best + slack(a, s);
            }
            settled = (settled && at[0] == at[1]) || s == 0.0f;        // (a zero takes the first level: every cost is lambda's part alone, or a NaN)
            if (active[e] && settled) {
#pragma unroll
                for (int k = 0; k < K; ++k) cnt[k] += at[0] == k;
            }
            bool keep = active[e] && !settled;
            unsigned long long m = __ballot(keep);
            if constexpr (COLLECT) {
                // equal scores stay open down to the last halving: those of a wavefront that equal its first one's travel as one entry
                // (a row of a few values would otherwise list itself)
#pragma unroll 1
                for (int r = 0; r < 2 && m != 0ull; ++r) {
                    const int leader = __ffsll((long long)m) - 1;
                    const float v = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(s), leader));
                    const unsigned long long same = __ballot(keep && s == v);
                    if (lane == leader) {
                        const int at = atomicAdd(&n_open, 1);
                        list[at] = v;
                        list_n[at] = (uint8_t)__popcll(same);
                    }
                    keep = keep && !(s == v);
                    m &= ~same;
                }
                if (m != 0ull) {
                    int at = 0;
                    if (lane == 0) at = atomicAdd(&n_open, __popcll(m));
                    at = __builtin_amdgcn_readfirstlane(at) + __popcll(m & ((1ull << lane) - 1ull));
                    if (keep) { list[at] = s; list_n[at] = 1; }
                }
            } else if (m != 0ull) {                                      // (wave-uniform)
                int at = 0;
                if (lane == 0) at = atomicAdd(&n_open, __popcll(m));
                at = __builtin_amdgcn_readfirstlane(at);
                if (keep) open[at + __popcll(m & ((1ull << lane) - 1ull))] = s;
            }
        }
        if (it + 1 < iters) request(it + 1);
        if constexpr (!COLLECT) {
            __syncthreads();
            const int count = n_open;
            __syncthreads();                                             // (nobody adds to it before everybody has read it)
            if (it + 1 == iters || count > LIST - RUN) {                 // (workgroup-uniform) no room for another run
                evaluate(count);
                __syncthreads();
                if (tid == 0) n_open = 0;
                __syncthreads();
            }
        }
    }
    if constexpr (COLLECT) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int s = wave_sum_dpp(cnt[k]);
            if (lane == 0 && s) atomicAdd(&lsum[k], (unsigned int)s);
        }
    } else {
        int settled_sum = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) settled_sum += cnt[k] * a.nominal[k];
        settled_sum = wave_sum_dpp(settled_sum);
#pragma unroll
        for (int o = NGRID; o < 64; o <<= 1) {
            sum += (unsigned int)__shfl_xor((int)sum, o, WAVE);
            ties += (unsigned int)__shfl_xor((int)ties, o, WAVE);
        }
        if (lane < NGRID) {
            atomicAdd(&lsum[lane], sum + (unsigned int)settled_sum);
            if (ties) atomicAdd(&lsum[NGRID + lane], ties);
        }
    }
    __syncthreads();
    unsigned int* mine = a.partial + (((size_t)(COLLECT ? a.rows : 0) + row) * a.n_chunks + blockIdx.x) * SLOTS;
    if (tid < SLOTS) mine[tid] = COLLECT && tid == NLV ? (unsigned int)n_open : lsum[tid];
}

// ---- the replay ----
// FN_OPEN entries of the list are kept in LDS; a longer one is read from memory every time.  Up to a row a compute unit, a workgroup has eight
// wavefronts (two a SIMD: sixteen got in the way of the replay's scalar steps) and room for 16384; 84 KB and 143 registers leave
// a compute unit to one row at a time, so that a call of more rows takes four wavefronts and room for 4096 (23 KB), four rows and more at a time.  us a call,
// eight wavefronts and 16384 / these: 300 rows of 128 scores 88 / 73, 1024 160 / 110, 4096 561 / 360 (two wavefronts and 2048: 324), 2048 of
// 20000 692 / 598; lists beyond the room (512 rows of 20000 scores that are nearly equal) 851 / 837 (two and 2048: 880).
#define FN_ROWS 256
template <int K, int FN_THREADS, int FN_OPEN>
__global__ __launch_bounds__(FN_THREADS) void alloc_finish_kernel(AllocArgs a) {
    constexpr int FN_WAVES = FN_THREADS / 64;
    __shared__ RowState cur;
    __shared__ float open[FN_OPEN];
    __shared__ uint8_t open_n[FN_OPEN];
    __shared__ int at[EV_MAX_CHUNKS + 1];                    // where a chunk's entries begin
    __shared__ int left[EV_MAX_CHUNKS];
    __shared__ int settled[NLV], hist[NLV];
    __shared__ int red[2][FN_WAVES];
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const RowState* in = a.state + row;
    const unsigned int* part = a.partial + ((size_t)a.rows + row) * a.n_chunks * SLOTS;
    unsigned int v[EV_MAX_CHUNKS * SLOTS / FN_THREADS];
    const int n_part = a.n_chunks * SLOTS;
#pragma unroll
    for (int u = 0; u < EV_MAX_CHUNKS * SLOTS / FN_THREADS; ++u) v[u] = tid + u * FN_THREADS < n_part ? part[tid + u * FN_THREADS] : 0u;
    if (tid == 0) cur = *in;
    if (tid < NLV) { settled[tid] = 0; hist[tid] = 0; }
    for (int i = tid; i <= EV_MAX_CHUNKS; i += FN_THREADS) at[i] = 0;
    __syncthreads();
    if (cur.n_active == 0) {
        if (tid == 0) a.state[(size_t)a.rows + row] = cur;
        return;
    }
#pragma unroll
    for (int u = 0; u < EV_MAX_CHUNKS * SLOTS / FN_THREADS; ++u) {
        const int e = tid + u * FN_THREADS, slot = e & (SLOTS - 1);
        if (e < n_part && slot < NLV && v[u]) atomicAdd(&settled[slot], (int)v[u]);
        if (e < n_part && slot == NLV) at[e / SLOTS + 1] = (int)v[u];
    }
    __syncthreads();
    auto running_sum = [&] {                                 // of at[], by the first wavefront: four chunks a lane
        if (wave != 0) return;
        static_assert(EV_MAX_CHUNKS == 256, "four chunks a lane");
        int mine[4], tot = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) { mine[i] = at[4 * lane + i + 1]; tot += mine[i]; }
        int incl = tot;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(incl, o, WAVE);
            if (lane >= o) incl += up;
        }
        int run = incl - tot;
#pragma unroll
        for (int i = 0; i < 4; ++i) { run += mine[i]; at[4 * lane + i + 1] = run; }
    };
    running_sum();
    __syncthreads();
    int n_open = at[a.n_chunks];
    bool in_lds = n_open <= FN_OPEN;
    float* list = a.open + (size_t)row * a.n;
    uint8_t* list_n = a.open_n + (size_t)row * a.n;
    auto fetch = [&] {
        // an entry per thread, whichever chunk it is from: one round trip for them all (a chunk per wavefront was one each)
        for (int i = tid; i < n_open; i += FN_THREADS) {
            int ch = 0;                                      // the last chunk that begins at or before i
#pragma unroll
            for (int step = EV_MAX_CHUNKS / 2; step >= 1; step >>= 1)
                if (ch + step < a.n_chunks && at[ch + step] <= i) ch += step;
            const size_t src = (size_t)ch * a.chunk_tokens + (i - at[ch]);
            open[i] = list[src];
            open_n[i] = list_n[src];
        }
    };
    if (in_lds) fetch();
    __syncthreads();
    // calls visit(score, tokens) for every entry, shared out over the workgroup
    auto walk = [&](auto visit) {
        if (in_lds) {
            for (int i = tid; i < n_open; i += FN_THREADS) visit(open[i], (int)open_n[i]);
        } else {
            for (int ch = wave; ch < a.n_chunks; ch += FN_WAVES) {
                const int n = at[ch + 1] - at[ch];
                const float* lp = list + (size_t)ch * a.chunk_tokens;
                const uint8_t* np = list_n + (size_t)ch * a.chunk_tokens;
                for (int i = lane; i < n; i += 4 * 64) {     // four reads under way
                    float s[4];
                    int c[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) { s[u] = i + 64 * u < n ? lp[i + 64 * u] : 0.0f; c[u] = i + 64 * u < n ? (int)np[i + 64 * u] : 0; }
#pragma unroll
                    for (int u = 0; u < 4; ++u) visit(s[u], c[u]);
                }
            }
        }
    };
    auto level = [&](float s, const float* lb) {
        float bc = __fadd_rn(__fmul_rn(s, a.eps[0]), lb[0]);
        int best = 0;
#pragma unroll
        for (int k = 1; k < K; ++k) {
            const float cst = __fadd_rn(__fmul_rn(s, a.eps[k]), lb[k]);
            if (cst < bc) { bc = cst; best = k; }
        }
        return best;
    };
    int settled_sum = 0;
    for (int k = 0; k < K; ++k) settled_sum += settled[k] * a.nominal[k];
    const float la = cur.la, lb = cur.lb, nf = (float)cur.n_active;
    const double target = cur.target;
    float known_above = -1.0f, known_within = -1.0f;         // the last two multipliers that were summed: later ones round to them
    int turn = 0;
    int asked = 0;
    // A list that does not fit LDS (scores within a thousandth of each other, all different): after every third sum, an eighth of the bracket
    // later, the tokens that are settled by now are counted and the others closed up, chunk by chunk where they lie, until it fits.
    auto close_up = [&] {
        const float from = fmaxf(cur.wa, known_above), to = known_within < 0.0f ? lb : fminf(lb, known_within);
        float c0[K], c1[K];
        int cnt[K];
#pragma unroll
        for (int k = 0; k < K; ++k) { c0[k] = __fmul_rn(from, a.bitsf[k]); c1[k] = __fmul_rn(to, a.bitsf[k]); cnt[k] = 0; }
#pragma unroll 1
        for (int ch = wave; ch < a.n_chunks; ch += FN_WAVES) {
            const int n = at[ch + 1] - at[ch];
            float* lp = list + (size_t)ch * a.chunk_tokens;
            uint8_t* np = list_n + (size_t)ch * a.chunk_tokens;
            int w = 0;                                       // (entries are written at or before the place they were read from, by the same wavefront)
            for (int i0 = 0; i0 < n; i0 += 64) {
                const bool on = i0 + lane < n;
                const float s = on ? lp[i0 + lane] : 0.0f;
                const int tokens = on ? (int)np[i0 + lane] : 0;
                float p0 = __fadd_rn(__fmul_rn(s, a.eps[0]), c0[0]), p1 = __fadd_rn(__fmul_rn(s, a.eps[0]), c1[0]), q0 = INFINITY, q1 = INFINITY;
                int b0 = 0, b1 = 0;
#pragma unroll
                for (int k = 1; k < K; ++k) {
                    const float se = __fmul_rn(s, a.eps[k]), v0 = __fadd_rn(se, c0[k]), v1 = __fadd_rn(se, c1[k]);
                    q0 = __builtin_amdgcn_fmed3f(v0, p0, q0);
                    q1 = __builtin_amdgcn_fmed3f(v1, p1, q1);
                    if (v0 < p0) { p0 = v0; b0 = k; }
                    if (v1 < p1) { p1 = v1; b1 = k; }
                }
                const bool is_settled = b0 == b1 && q0 * KEEP > p0 + slack(a, s) && q1 * KEEP > p1 + slack(a, s);
#pragma unroll
                for (int k = 0; k < K; ++k) cnt[k] += is_settled && b0 == k ? tokens : 0;
                const bool keep = on && !is_settled;
                const unsigned long long m = __ballot(keep);
                if (keep) {
                    const int at_ = w + __popcll(m & ((1ull << lane) - 1ull));
                    lp[at_] = s;
                    np[at_] = (uint8_t)tokens;
                }
                w += __popcll(m);
            }
            if (lane == 0) left[ch] = w;
        }
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int s = wave_sum_int(cnt[k]);
            if (lane == 0 && s) atomicAdd(&settled[k], s);
        }
        __syncthreads();                                     // everybody has read where its chunks began
        for (int i = tid; i < EV_MAX_CHUNKS; i += FN_THREADS) at[i + 1] = i < a.n_chunks ? left[i] : 0;     // (the old sums behind the last chunk must not be summed again)
        __syncthreads();
        running_sum();
        __syncthreads();
        n_open = at[a.n_chunks];
        in_lds = n_open <= FN_OPEN;
        if (in_lds) fetch();                                 // (other wavefronts' entries: the barriers above order their stores)
        settled_sum = 0;
        for (int k = 0; k < K; ++k) settled_sum += settled[k] * a.nominal[k];
        __syncthreads();
    };
    const bool may_close = cur.wa == fmaxf(la, LAMBDA_LEAST) && cur.wb == lb;     // (else the final multiplier may lie beside the window)
    const double lam = replay(lb, [&](float lambda) {            // (every thread runs it: the answers are the workgroup's)
        if (lambda <= la || lambda == known_above) return true;
        if (lambda >= lb || lambda == known_within) return false;
        if (!in_lds && may_close && asked > 0 && asked % 3 == 0) close_up();
        ++asked;
        float cost[K];
#pragma unroll
        for (int k = 0; k < K; ++k) cost[k] = __fmul_rn(lambda, a.bitsf[k]);
        int sum = 0;
        walk([&](float s, int n) {
            float bc = __fadd_rn(__fmul_rn(s, a.eps[0]), cost[0]);
            int bn = a.nominal[0];
#pragma unroll
            for (int k = 1; k < K; ++k) {
                const float cst = __fadd_rn(__fmul_rn(s, a.eps[k]), cost[k]);
                if (cst < bc) { bc = cst; bn = a.nominal[k]; }
            }
            sum += bn * n;
        });
        sum = wave_sum_dpp(sum);
        if (lane == 0) red[turn][wave] = sum;
        __syncthreads();                                     // (one barrier a sum: the next one writes the other half)
        int all = settled_sum;
#pragma unroll
        for (int w = 0; w < FN_WAVES; ++w) all += red[turn][w];
        turn ^= 1;
        const bool above = (double)((float)all / nf) > target;
        if (above) known_above = lambda; else known_within = lambda;
        return above;
    });
    float cost[K];
#pragma unroll
    for (int k = 0; k < K; ++k) cost[k] = __fmul_rn((float)lam, a.bitsf[k]);
    int cnt[K];
#pragma unroll
    for (int k = 0; k < K; ++k) cnt[k] = 0;
    walk([&](float s, int n) {
        const int best = level(s, cost);
#pragma unroll
        for (int k = 0; k < K; ++k) cnt[k] += best == k ? n : 0;
    });
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int s = wave_sum_int(cnt[k]);
        if (lane == 0 && s) atomicAdd(&hist[k], s);
    }
    __syncthreads();
    if (tid == 0) {
        unsigned long long S = 0ull;
        for (int k = 0; k < K; ++k) {
            cur.final_hist[k] = settled[k] + hist[k];
            S += (unsigned long long)cur.final_hist[k] * (unsigned long long)a.nominal[k];
        }
        const double avg = (double)((float)S / nf);
        cur.gap = (avg - target) * (double)cur.n_active;
        cur.lam = lam;
        a.state[(size_t)a.rows + row] = cur;
        if (a.lambda_out) a.lambda_out[row] = lam;
    }
}

// ---- budget repair -------------------------------------------------------------------------------
// The host formulation sorts the row by score (stable) and, walking the level pairs, moves the
// n lowest-scored tokens of the upper level down (over budget) or the n highest-scored tokens of the
// lower level up (under budget).  Equivalent without a sort: among the tokens at level `from`,
// take the n smallest (largest) 64-bit keys (score bits, index).
struct Move { int from, to, want, i; bool lowest; double delta; };

// the first level pair, at or after pair index i in walking order, that moves tokens
__device__ static inline bool next_move(const AllocArgs& a, const int* hist, double gap_abs, bool over, int i, Move& m) {
    for (; over ? i < a.K - 1 : i >= 0; i += over ? 1 : -1) {
        const double delta = (double)a.bitsf[i + 1] - (double)a.bitsf[i];
        if (delta <= 0) continue;
        const int have = over ? hist[i + 1] : hist[i];
        const int n = min(have, (int)(gap_abs / delta + 0.5));
        if (n <= 0) continue;
        m.from = over ? i + 1 : i; m.to = over ? i : i + 1; m.want = n; m.i = i; m.lowest = over; m.delta = delta;
        return true;
    }
    return false;
}

__device__ static inline unsigned long long token_key(float s, int i, bool lowest) {
    // + 1 keeps both k and ~k away from the "no key" value
    const unsigned long long k = (((unsigned long long)__float_as_uint(s) << 32) | (unsigned int)i) + 1ull;
    return lowest ? k : ~k;            // always select minima
}
__device__ static inline unsigned int key_index(unsigned long long g, bool lowest) {
    return (unsigned int)(((lowest ? g : ~g) - 1ull) & 0xffffffffull);
}

__device__ static inline unsigned long long wave_min_u64(unsigned long long v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const unsigned long long other = __shfl_xor(v, o, WAVE);
        v = other < v ? other : v;
    }
    return v;
}

#define KEY_NONE 0xffffffffffffffffull

// `want` rounds of a workgroup-wide minimum over the keys held in registers; every selected key is
// handed to `emit(round, key)` by thread 0 and struck from its owner's registers
template <int NK, int NWAVES, typename F>
__device__ static inline void select_smallest(unsigned long long (&keys)[NK], int want, unsigned long long* wbest, F emit) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    for (int r = 0; r < want; ++r) {
        unsigned long long best = KEY_NONE;
#pragma unroll
        for (int e = 0; e < NK; ++e) best = keys[e] < best ? keys[e] : best;
        const unsigned long long wb = wave_min_u64(best);
        if (lane == 0) wbest[wave] = wb;
        __syncthreads();
        unsigned long long g = KEY_NONE;
        for (int w = 0; w < NWAVES; ++w) g = wbest[w] < g ? wbest[w] : g;
        if (g != KEY_NONE) {
#pragma unroll
            for (int e = 0; e < NK; ++e) keys[e] = keys[e] == g ? KEY_NONE : keys[e];
        }
        if (tid == 0) emit(r, g);
        __syncthreads();
    }
}

// Levels at the final multiplier, and per chunk the candidates for the repair's moves that are small.  (A move takes tokens from a level
// that no earlier move of the walk has touched, so all of them are chosen from the levels as they are.)
template <int K>
__global__ __launch_bounds__(EV_THREADS) void alloc_assign_kernel(AllocArgs a) {
    __shared__ unsigned long long wbest[EV_THREADS / 64];
    __shared__ RowState cur;
    const int row = blockIdx.y, tid = threadIdx.x;
    const int base = blockIdx.x * EV_TOKENS;
    float score[EV_TPT];
    bool on[EV_TPT];
#pragma unroll
    for (int e = 0; e < EV_TPT; ++e) {
        const int i = base + e * EV_THREADS + tid;
        on[e] = i < a.n && !is_sink(a, row, i);
        score[e] = on[e] ? a.scores[(size_t)row * a.n + i] : 0.0f;
    }
    if (tid == 0) cur = a.state[(size_t)a.rows + row];
    __syncthreads();
    const RowState& st = cur;
    const Cleaner clean(st);
    float cost[K];
#pragma unroll
    for (int k = 0; k < K; ++k) cost[k] = __fmul_rn((float)st.lam, a.bitsf[k]);
    int level[EV_TPT];
#pragma unroll
    for (int e = 0; e < EV_TPT; ++e) {
        const int i = base + e * EV_THREADS + tid;
        level[e] = -1;
        int out = a.sink_bits;
        if (on[e]) {
            score[e] = clean(score[e]);
            float bc = __fadd_rn(__fmul_rn(score[e], a.eps[0]), cost[0]);
            int best = 0;
            out = a.nominal[0];
#pragma unroll
            for (int k = 1; k < K; ++k) {
                const float cst = __fadd_rn(__fmul_rn(score[e], a.eps[k]), cost[k]);
                if (cst < bc) { bc = cst; best = k; out = a.nominal[k]; }
            }
            level[e] = best;
        }
        if (i < a.n) a.bits_out[(size_t)row * a.n + i] = out;
    }
    if (st.n_active == 0 || fabs(st.gap) <= 0.5) return;
    const bool over = st.gap > 0;
    double gap = fabs(st.gap);
    unsigned long long* out = a.cand + ((size_t)row * a.n_cand + blockIdx.x) * NLV * CAND_MAX;
    int i = over ? 0 : a.K - 2;
    Move m;
    for (int j = 0; next_move(a, st.final_hist, gap, over, i, m); ++j) {                  // the walk of alloc_repair_kernel
        if (m.want <= CAND_MAX) {
            unsigned long long keys[EV_TPT];
#pragma unroll
            for (int e = 0; e < EV_TPT; ++e)
                keys[e] = level[e] == m.from ? token_key(score[e], base + e * EV_THREADS + tid, m.lowest) : KEY_NONE;
            select_smallest<EV_TPT, EV_THREADS / 64>(keys, m.want, wbest, [&](int r, unsigned long long g) { out[j * CAND_MAX + r] = g; });
        }
        gap -= m.want * m.delta;
        if (gap <= 0.5) break;
        i = m.i + (over ? 1 : -1);
    }
}

#define RB 1024
#define MV_TPT 8

// Moves `want` tokens currently at width `from` to width `to`: those with the smallest
// (score, index) if lowest, else those with the largest.  Scores are non-negative and finite,
// so their bit patterns order like the values.
__device__ static void move_tokens(const AllocArgs& a, int row, const Cleaner& clean, int from, int to, int want,
                                   bool lowest, unsigned int* hist256, int* scratch) {
    const float* s = a.scores + (size_t)row * a.n;
    int32_t* ch = a.bits_out + (size_t)row * a.n;
    const int tid = threadIdx.x;
    // calls visit(index, key) for every token at `from`, eight reads of a thread under way (one at a time the passes were a
    // chain of round trips: 262144 equal scores 1.44 ms a call, 1.14 now)
    auto walk = [&](auto visit) {
        for (int i0 = tid; i0 < a.n; i0 += MV_TPT * RB) {
            float v[MV_TPT];
            int at[MV_TPT];
#pragma unroll
            for (int u = 0; u < MV_TPT; ++u) {
                const int i = i0 + u * RB;
                at[u] = i < a.n ? ch[i] : -1;
                v[u] = i < a.n ? s[i] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < MV_TPT; ++u)
                if (at[u] == from && !is_sink(a, row, i0 + u * RB)) visit(i0 + u * RB, __float_as_uint(clean(v[u])));
        }
    };
    // radix select, most significant byte first: find the key of the want-th token
    unsigned int prefix = 0u, pmask = 0u;
    int remaining = want;       // rank still to find inside the current prefix class
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        for (int e = tid; e < 256; e += RB) hist256[e] = 0u;
        __syncthreads();
        walk([&](int, unsigned int key) {
            if ((key & pmask) == prefix) atomicAdd(&hist256[(key >> shift) & 0xffu], 1u);
        });
        __syncthreads();
        if (tid == 0) {
            int acc = 0, bin;
            if (lowest) {
                for (bin = 0; bin < 256; ++bin) { if (acc + (int)hist256[bin] >= remaining) break; acc += hist256[bin]; }
            } else {
                for (bin = 255; bin >= 0; --bin) { if (acc + (int)hist256[bin] >= remaining) break; acc += hist256[bin]; }
            }
            bin = bin < 0 ? 0 : (bin > 255 ? 255 : bin);
            scratch[0] = bin;
            scratch[1] = remaining - acc;
        }
        __syncthreads();
        prefix |= ((unsigned int)scratch[0]) << shift;
        pmask |= 0xffu << shift;
        remaining = scratch[1];
        __syncthreads();
    }
    // `prefix` is the threshold key; `remaining` of the tokens equal to it move, in index order
    // (the first ones if lowest, the last ones otherwise)
    if (tid == 0) scratch[2] = 0;      // ties seen so far
    if (!lowest) {
        // count the ties to know how many to skip
        if (tid == 0) scratch[3] = 0;
        __syncthreads();
        int local = 0;
        walk([&](int, unsigned int key) { local += key == prefix; });
        if (local) atomicAdd(&scratch[3], local);
        __syncthreads();
    }
    __syncthreads();
    const int n_eq = lowest ? 0 : scratch[3];
    const int first_tie = lowest ? 0 : n_eq - remaining;          // ties with rank in [first_tie, first_tie + remaining) move
    const int wave = tid >> 6, lane = tid & 63;
    int* wave_cnt = scratch + 8;                                  // [16]
    for (int c = 0; c < a.n; c += MV_TPT * RB) {                  // a wavefront takes MV_TPT x 64 tokens behind one another
        const int i0 = c + wave * (MV_TPT * 64) + lane;
        float v[MV_TPT];
        int at[MV_TPT];
#pragma unroll
        for (int u = 0; u < MV_TPT; ++u) {
            const int i = i0 + u * 64;
            at[u] = i < a.n ? ch[i] : -1;
            v[u] = i < a.n ? s[i] : 0.0f;
        }
        unsigned long long ties[MV_TPT];
        bool strict[MV_TPT];
        int n_ties = 0;
#pragma unroll
        for (int u = 0; u < MV_TPT; ++u) {
            const bool member = at[u] == from && !is_sink(a, row, i0 + u * 64);
            const unsigned int key = __float_as_uint(clean(v[u]));
            strict[u] = member && (lowest ? key < prefix : key > prefix);
            ties[u] = __ballot(member && key == prefix);
            n_ties += __popcll(ties[u]);
        }
        if (lane == 0) wave_cnt[wave] = n_ties;
        __syncthreads();
        int before = scratch[2];
        for (int w = 0; w < wave; ++w) before += wave_cnt[w];
#pragma unroll
        for (int u = 0; u < MV_TPT; ++u) {
            const int rank = before + __popcll(ties[u] & ((1ull << lane) - 1ull));
            const bool tie = (ties[u] >> lane) & 1ull;
            if (strict[u] || (tie && rank >= first_tie && rank < first_tie + remaining)) ch[i0 + u * 64] = to;
            before += __popcll(ties[u]);
        }
        __syncthreads();
        if (tid == 0) {
            int tot = 0;
            for (int w = 0; w < RB / 64; ++w) tot += wave_cnt[w];
            scratch[2] += tot;
        }
        __syncthreads();
    }
}

// one workgroup per row: apply the moves from the chunk candidates where they are small, the others by a radix select over
// the row (a pass of one workgroup over all of it, five times: 4.4 ms for a million equal scores; while only the first move had
// candidates, and only up to 4096 of them, one row in four of that length took it)
__global__ __launch_bounds__(RB) void alloc_repair_kernel(AllocArgs a) {
    __shared__ unsigned int hist256[256];
    __shared__ int scratch[32];
    __shared__ unsigned long long wbest[RB / 64];
    const int row = blockIdx.x, tid = threadIdx.x;
    const RowState& st = a.state[(size_t)a.rows + row];
    if (st.n_active == 0) return;                            // (its counts are the cleared ones)
    if (a.level_counts && tid < a.K) a.level_counts[row * a.K + tid] = st.final_hist[tid];
    double gap = st.gap;
    if (fabs(gap) <= 0.5) return;
    __syncthreads();                                         // thread 0 moves counts below
    const bool over = gap > 0;
    gap = fabs(gap);
    const Cleaner clean(st);
    int i = over ? 0 : a.K - 2;
    Move m;
    int32_t* ch = a.bits_out + (size_t)row * a.n;
    for (int j = 0; next_move(a, st.final_hist, gap, over, i, m); ++j) {
        const unsigned long long* cand = a.cand + ((size_t)row * a.n_cand * NLV + j) * CAND_MAX;
        const int total = a.n_cand * m.want;
        auto key_at = [&](int idx) { return idx < total ? cand[(size_t)(idx / m.want) * (NLV * CAND_MAX) + idx % m.want] : KEY_NONE; };
        auto move = [&](int, unsigned long long g) { if (g != KEY_NONE) ch[key_index(g, m.lowest)] = a.nominal[m.to]; };
        if (m.want <= CAND_MAX && total <= 4 * RB) {
            unsigned long long keys[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) keys[e] = key_at(e * RB + tid);
            select_smallest<4, RB / 64>(keys, m.want, wbest, move);
        } else if (m.want <= CAND_MAX && total <= 16 * RB) {
            unsigned long long keys[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) keys[e] = key_at(e * RB + tid);
            select_smallest<16, RB / 64>(keys, m.want, wbest, move);
        } else {
            __syncthreads();
            move_tokens(a, row, clean, a.nominal[m.from], a.nominal[m.to], m.want, m.lowest, hist256, scratch);
        }
        if (tid == 0 && a.level_counts) {
            a.level_counts[row * a.K + m.from] -= m.want;
            a.level_counts[row * a.K + m.to] += m.want;
        }
        gap -= m.want * m.delta;
        if (gap <= 0.5) break;
        i = m.i + (over ? 1 : -1);
    }
}

// a single level: nothing to choose
__global__ __launch_bounds__(EV_THREADS) void alloc_write_kernel(AllocArgs a) {
    __shared__ int n_level;
    const int row = blockIdx.y;
    if (threadIdx.x == 0) n_level = 0;
    __syncthreads();
    const int base = blockIdx.x * EV_TOKENS;
    for (int e = 0; e < EV_TPT; ++e) {
        const int i = base + e * EV_THREADS + threadIdx.x;
        const bool on = i < a.n && !is_sink(a, row, i);
        if (i < a.n) a.bits_out[(size_t)row * a.n + i] = on ? a.nominal[0] : a.sink_bits;
        const int n = __popcll(__ballot(on));
        if ((threadIdx.x & 63) == 0 && n) atomicAdd(&n_level, n);
    }
    __syncthreads();
    if (a.level_counts && threadIdx.x == 0 && n_level) atomicAdd(&a.level_counts[row * a.K], n_level);
}

struct AllocLayout { size_t range, hist, partial, open, open_n, cand, state, total; };
static AllocLayout alloc_layout(int rows, int n) {
    AllocLayout L;
    rows = std::min(rows, MAX_TURN);
    const size_t chunks = ((size_t)n + EV_TOKENS - 1) / EV_TOKENS, evals = ((size_t)n + EV_THREADS - 1) / EV_THREADS;
    size_t off = 0;
    auto take = [&](size_t bytes) { size_t o = off; off += align_up(bytes, 256); return o; };
    L.range = take((size_t)rows * (((size_t)n + SC_THREADS * SC_SMALL - 1) / (SC_THREADS * SC_SMALL)) * sizeof(uint2));
    L.hist = take((size_t)rows * HB_BINS * sizeof(unsigned int));
    L.partial = take((size_t)2 * rows * std::min<size_t>(evals, EV_MAX_CHUNKS) * SLOTS * sizeof(unsigned int));
    L.open = take((size_t)rows * n * sizeof(float));
    L.open_n = take((size_t)rows * n);
    L.cand = take((size_t)rows * chunks * NLV * CAND_MAX * sizeof(unsigned long long));
    L.state = take((size_t)2 * rows * sizeof(RowState));
    L.total = off;
    return L;
}

extern "C" size_t odmkv_allocate_workspace_bytes(int rows, int n) {
    if (rows <= 0 || n <= 0) return 0;
    return alloc_layout(rows, n).total;
}

template <int K>
static int launch_search(const AllocArgs& a, int tpt, hipStream_t st) {
    const dim3 grid(a.n_chunks, a.rows), block(EV_THREADS);
    hipLaunchKernelGGL(alloc_search_kernel, dim3(a.rows), dim3(SE_THREADS), 0, st, a);
    ODMKV_CHECK_LAUNCH("alloc_search_kernel");
    if (tpt == 1) hipLaunchKernelGGL((alloc_pass_kernel<K, 1, false>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((alloc_pass_kernel<K, EV_BIG, false>), grid, block, 0, st, a);
    ODMKV_CHECK_LAUNCH("alloc_pass_kernel (narrow)");
    if (tpt == 1) hipLaunchKernelGGL((alloc_pass_kernel<K, 1, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((alloc_pass_kernel<K, EV_BIG, true>), grid, block, 0, st, a);
    ODMKV_CHECK_LAUNCH("alloc_pass_kernel (collect)");
    if (a.rows <= FN_ROWS) hipLaunchKernelGGL((alloc_finish_kernel<K, 512, 16384>), dim3(a.rows), dim3(512), 0, st, a);
    else hipLaunchKernelGGL((alloc_finish_kernel<K, 256, 4096>), dim3(a.rows), dim3(256), 0, st, a);
    ODMKV_CHECK_LAUNCH("alloc_finish_kernel");
    hipLaunchKernelGGL((alloc_assign_kernel<K>), dim3(a.n_cand, a.rows), block, 0, st, a);
    ODMKV_CHECK_LAUNCH("alloc_assign_kernel");
    hipLaunchKernelGGL(alloc_repair_kernel, dim3(a.rows), dim3(RB), 0, st, a);
    ODMKV_CHECK_LAUNCH("alloc_repair_kernel");
    return 0;
}

extern "C" int odmkv_allocate(const float* scores, int rows, int n,
                              const uint8_t* sink_mask, int period, int n_sink, int sink_bits,
                              const int32_t* levels, int n_levels, const double* eps,
                              const double* target,
                              int32_t* bits_out, int32_t* level_counts, double* lambda_out,
                              void* workspace, size_t workspace_bytes, void* stream) {
    ODMKV_CHECK_ARG(scores && levels && eps && target && bits_out && workspace, "allocate: null pointer");
    ODMKV_CHECK_ARG(rows > 0 && n > 0, "allocate: bad shape rows=%d n=%d", rows, n);
    ODMKV_CHECK_ARG(n_levels >= 1 && n_levels <= NLV, "allocate: between 1 and %d levels, got %d", NLV, n_levels);
    for (int k = 0; k < n_levels; ++k) {
        ODMKV_CHECK_ARG(levels[k] >= 0 && levels[k] <= 16, "allocate: level %d out of range", levels[k]);
        ODMKV_CHECK_ARG(k == 0 || levels[k] > levels[k - 1], "allocate: levels must be strictly ascending");
    }
    ODMKV_CHECK_ARG(sink_mask || n_sink == 0 || (period > 0 && n % period == 0 && n_sink <= period),
                    "allocate: bad sink pattern period=%d n_sink=%d n=%d", period, n_sink, n);
    // bit sums up to 2^24 are exact in fp32, which the fp32 mean of the host formulation relies on
    ODMKV_CHECK_ARG((double)n * 16.0 <= 16777216.0, "allocate: rows longer than 1,048,576 tokens lose exactness of the fp32 mean");
    ODMKV_CHECK_ARG(rows <= 65535, "allocate: at most 65535 rows per call");
    ODMKV_CHECK_ARG(workspace_bytes >= odmkv_allocate_workspace_bytes(rows, n), "allocate: workspace too small");
    hipStream_t st = (hipStream_t)stream;
    const AllocLayout L = alloc_layout(rows, n);
    char* ws = (char*)workspace;
    AllocArgs a;
    a.n = n;
    a.period = period > 0 ? period : n; a.n_sink = sink_mask ? 0 : n_sink; a.sink_bits = sink_bits; a.K = n_levels;
    a.n_cand = (n + EV_TOKENS - 1) / EV_TOKENS;
    for (int k = 0; k < NLV; ++k) {
        a.eps[k] = k < n_levels ? (float)eps[k] : 0.0f;
        a.bitsf[k] = k < n_levels ? (float)levels[k] : 0.0f;
        a.nominal[k] = k < n_levels ? levels[k] : 0;
    }
    // A NaN or infinite error means the same for every positive score at every multiplier, and a zero score takes the first level whatever
    // the table says (its product is a NaN, or it costs least): the first level's NaN, which keeps every token, is -inf; another's, never
    // below anything, and -inf behind -inf, never below that, are +inf.
    bool seen_lowest = false;
    float negative = 0.0f;
    for (int k = 0; k < n_levels; ++k) {
        if (std::isnan(a.eps[k])) a.eps[k] = k == 0 ? -INFINITY : INFINITY;
        if (a.eps[k] == -INFINITY && seen_lowest) a.eps[k] = INFINITY;
        seen_lowest = seen_lowest || a.eps[k] == -INFINITY;
        if (std::isfinite(a.eps[k])) negative = std::max(negative, -a.eps[k]);
    }
    a.slack_s = 0x1p-18f * negative;
    a.n_steps = 0;
    a.first_bits = levels[0];
    for (int at = 0; at < n_levels - 1;) {
        int next = -1;
        double ratio = INFINITY;                                         // score / lambda from which `next` is better than `at`
        for (int k = at + 1; k < n_levels; ++k) {
            const double gain = (double)a.eps[at] - (double)a.eps[k];
            const double r = gain > 0.0 ? (levels[k] - levels[at]) / gain : INFINITY;
            if ((r < ratio || (r == ratio && r > 0.0)) && r < 1e30) { ratio = r; next = k; }      // (out of an infinite error: the narrowest finite one)
        }
        if (next < 0) break;
        a.step_at[a.n_steps] = (float)ratio;
        a.step_bits[a.n_steps++] = (float)(levels[next] - levels[at]);
        at = next;
    }
    a.range = (uint2*)(ws + L.range);
    a.hist = (unsigned int*)(ws + L.hist);
    a.partial = (unsigned int*)(ws + L.partial);
    a.open = (float*)(ws + L.open);
    a.open_n = (uint8_t*)(ws + L.open_n);
    a.cand = (unsigned long long*)(ws + L.cand);
    a.state = (RowState*)(ws + L.state);
    for (int r0 = 0; r0 < rows; r0 += MAX_TURN) {                        // (the workspace is a turn's; the stream orders the turns)
        a.rows = std::min(rows - r0, MAX_TURN);
        a.scores = scores + (size_t)r0 * n;
        a.sink_mask = sink_mask ? sink_mask + (size_t)r0 * n : nullptr;
        a.target = target + r0;
        a.bits_out = bits_out + (size_t)r0 * n;
        a.level_counts = level_counts ? level_counts + (size_t)r0 * n_levels : nullptr;
        a.lambda_out = lambda_out ? lambda_out + r0 : nullptr;
        // one token per thread up to a workgroup of them per compute unit; then EV_BIG tokens per thread and run, as many runs as
        // leave EV_WGS workgroups over all rows, two per compute unit
        const long long all = (long long)a.rows * n;
        const int tpt = all <= 256ll * EV_THREADS ? 1 : EV_BIG, run = EV_THREADS * tpt;
        const int runs = (n + run - 1) / run;
        a.iters = (int)std::max<long long>((runs + EV_MAX_CHUNKS - 1) / EV_MAX_CHUNKS, (all + EV_WGS * run - 1) / (EV_WGS * run));
        if (tpt == 1) a.iters = 1;
        a.iters = std::min(a.iters, runs);
        a.chunk_tokens = a.iters * run;
        a.n_chunks = (runs + a.iters - 1) / a.iters;
        const bool small = all <= 256ll * SC_THREADS * SC_SMALL;
        a.n_scan = small ? (n + SC_THREADS * SC_SMALL - 1) / (SC_THREADS * SC_SMALL) : (n + SC_THREADS * SC_BIG - 1) / (SC_THREADS * SC_BIG);
        const dim3 scan(a.n_scan, a.rows);
        if (small) hipLaunchKernelGGL(alloc_range_kernel<SC_SMALL>, scan, dim3(SC_THREADS), 0, st, a);
        else hipLaunchKernelGGL(alloc_range_kernel<SC_BIG>, scan, dim3(SC_THREADS), 0, st, a);
        ODMKV_CHECK_LAUNCH("alloc_range_kernel");
        if (n_levels == 1) {
            hipLaunchKernelGGL(alloc_write_kernel, dim3(a.n_cand, a.rows), dim3(EV_THREADS), 0, st, a);
            ODMKV_CHECK_LAUNCH("alloc_write_kernel");
            continue;
        }
        if (small) hipLaunchKernelGGL(alloc_scan_kernel<SC_SMALL>, scan, dim3(SC_THREADS), 0, st, a);
        else hipLaunchKernelGGL(alloc_scan_kernel<SC_BIG>, scan, dim3(SC_THREADS), 0, st, a);
        ODMKV_CHECK_LAUNCH("alloc_scan_kernel");
        int rc = 0;
        switch (n_levels) {
            case 2: rc = launch_search<2>(a, tpt, st); break;
            case 3: rc = launch_search<3>(a, tpt, st); break;
            case 4: rc = launch_search<4>(a, tpt, st); break;
            case 5: rc = launch_search<5>(a, tpt, st); break;
            case 6: rc = launch_search<6>(a, tpt, st); break;
            case 7: rc = launch_search<7>(a, tpt, st); break;
            default: rc = launch_search<8>(a, tpt, st); break;
        }
        if (rc) return rc;
    }
    return 0;
}
