// Small changes of a store that holds tokens: a block of exact tokens behind the others, the newest exact tokens dropped,
// everything from a position on cut off.
#include <algorithm>
#include "quant.h"

// ------------------------------------------------------------------------------------------------
// T new exact tokens per (sequence, kv-head).  Bound by latency: one launch writes the rows, a second moves the counts (the
// workgroups of a segment all have to see the old one).  Through the general append (counts, compaction, the quantisers with
// nothing to quantise, the gather) 29 tokens of 8 heads took 60 us of kernels and a read-back; here 6 us and none.
// ------------------------------------------------------------------------------------------------
struct AppendRowsArgs {
    odmkv_packed_t s;
    const uint16_t* k;
    const uint16_t* v;
    long long sB, sH, sTk, sTv;
    int T, pos;
};

__global__ __launch_bounds__(HD) void append_rows_kernel(AppendRowsArgs a) {
    const int bh = blockIdx.y, j = threadIdx.x;
    const int count = a.s.seg_count[4][bh], first = a.s.seg_tile[4][bh];
    const int cap = (a.s.seg_tile[4][bh + 1] - first) * TILE;
    const size_t src = (size_t)(bh / a.s.Hkv) * a.sB + (size_t)(bh % a.s.Hkv) * a.sH + j;
    for (int t = blockIdx.x; t < a.T; t += gridDim.x) {
        const int at = count + t;
        if (at >= cap) return;                                   // full: the host sized it too small
        const size_t tile = (size_t)first + at / TILE;
        const int slot = at % TILE;
        a.s.kexact[tile * TILE * HD + exact_k_index(slot, j)] = a.k[src + (size_t)t * a.sTk];
        a.s.vexact[tile * TILE * HD + exact_v_index(slot, j)] = a.v[src + (size_t)t * a.sTv];
        if (j == 0) a.s.pos[4][tile * TILE + slot] = a.pos + t;
    }
}

// the exact segments' counts moved by n (not below zero, not beyond the room)
__global__ __launch_bounds__(256) void move_exact_counts_kernel(odmkv_packed_t s, int nseg, int n) {
    const int bh = blockIdx.x * 256 + threadIdx.x;
    if (bh >= nseg) return;
    const int cap = (s.seg_tile[4][bh + 1] - s.seg_tile[4][bh]) * TILE;
    s.seg_count[4][bh] = min(max(s.seg_count[4][bh] + n, 0), cap);
}

static int check_exact(const odmkv_packed_t* s, const char* who) {
    ODMKV_CHECK_ARG(s && s->B > 0 && s->Hkv > 0, "%s: bad store", who);
    ODMKV_CHECK_ARG(s->kexact && s->vexact && s->seg_tile[4] && s->seg_count[4] && s->pos[4], "%s: store has no exact segments", who);
    return 0;
}

static int move_counts(const odmkv_packed_t* store, int n, void* stream) {
    const int nseg = store->B * store->Hkv;
    hipLaunchKernelGGL(move_exact_counts_kernel, dim3((nseg + 255) / 256), dim3(256), 0, (hipStream_t)stream, *store, nseg, n);
    ODMKV_CHECK_LAUNCH("move_exact_counts_kernel");
    return 0;
}

extern "C" int odmkv_append_exact_rows(const odmkv_packed_t* store, const void* k, const void* v, int T, int64_t stride_b,
                                       int64_t stride_h, int64_t stride_tk, int64_t stride_tv, int pos, void* stream) {
    ODMKV_CHECK_ARG(k && v && T > 0, "append_exact_rows: null pointer or no tokens");
    if (int rc = check_exact(store, "append_exact_rows")) return rc;
    ODMKV_CHECK_ARG(store->B * store->Hkv <= 65535, "append_exact_rows: at most 65535 (sequence, head) pairs");
    ODMKV_CHECK_ARG(stride_b >= 0 && stride_h >= 0 && stride_tk >= 0 && stride_tv >= 0, "append_exact_rows: negative strides");
    const AppendRowsArgs a = {*store, (const uint16_t*)k, (const uint16_t*)v, (long long)stride_b, (long long)stride_h,
                              (long long)stride_tk, (long long)stride_tv, T, pos};
    hipLaunchKernelGGL(append_rows_kernel, dim3(std::min(T, 1024), store->B * store->Hkv), dim3(HD), 0, (hipStream_t)stream, a);
    ODMKV_CHECK_LAUNCH("append_rows_kernel");
    return move_counts(store, T, stream);
}

extern "C" int odmkv_drop_exact_tail(const odmkv_packed_t* store, int n, void* stream) {
    ODMKV_CHECK_ARG(n > 0, "drop_exact_tail: n=%d", n);
    if (int rc = check_exact(store, "drop_exact_tail")) return rc;
    return move_counts(store, -n, stream);
}

// ------------------------------------------------------------------------------------------------
// every segment cut at a position: positions ascend inside a segment, so the survivors are a prefix, found by bisection
// (a thread per segment and level).  The new counts also go to the host's page-locked mirror: reading five levels of
// positions back and searching them there took 0.4 ms of a 32k-token layer.
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void truncate_kernel(odmkv_packed_t s, int nseg, int length, int32_t* counts) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= 5 * nseg) return;
    const int li = i / nseg, bh = i % nseg;
    int lo = 0, hi = s.seg_count[li][bh];
    const int32_t* pos = s.pos[li] + (size_t)s.seg_tile[li][bh] * TILE;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (pos[mid] < length) lo = mid + 1;
        else hi = mid;
    }
    s.seg_count[li][bh] = lo;
    counts[i] = lo;
}

extern "C" int odmkv_truncate(const odmkv_packed_t* store, int length, int32_t* counts, void* stream) {
    ODMKV_CHECK_ARG(store && counts && store->B > 0 && store->Hkv > 0 && length >= 0, "truncate: bad arguments");
    for (int li = 0; li < 5; ++li)
        ODMKV_CHECK_ARG(store->seg_tile[li] && store->seg_count[li] && store->pos[li], "truncate: missing tables of level %d", li);
    const int nseg = store->B * store->Hkv;
    hipLaunchKernelGGL(truncate_kernel, dim3((5 * nseg + 255) / 256), dim3(256), 0, (hipStream_t)stream, *store, nseg, length, counts);
    ODMKV_CHECK_LAUNCH("truncate_kernel");
    return 0;
}
