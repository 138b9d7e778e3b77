// A layer's bit levels on their way from the allocation to the store: counted, its protected tail set to 16 bits, and
// written down as the store's level map, in one pass; and the list of evicted positions.
#include <algorithm>
#include "common.h"

#define LV_THREADS 256
#define LV_CHUNK 4096           // tokens per workgroup: sixteen per thread
#define LV_MAX_ROWS 65532       // rows of a launch (its y index): the largest multiple of four, so that each starts as aligned as the first

// 6-bit counters of the six levels in one 64-bit word; a value that is no level adds nothing (as in pack.hip)
__device__ static inline unsigned long long count_of(int bits) {
    const int slot = level_slot(bits);
    return slot >= 0 ? 1ull << (6 * slot) : 0ull;
}

struct LevelsArgs {
    int32_t* bits;                       // [rows, T], the tail overwritten
    uint8_t* levels;                     // [rows, stride]: T levels, then 16s
    int32_t* counts;                     // [rows, chunks, 2, 6]: tokens in [lo, hi) as allocated, and all of them as stored
    long long stride;
    int T, lo, hi, tail, chunks;
    int vec;                             // every row of bits starts on a multiple of 16 bytes
};

// Bound by latency: 1 MB in, 0.26 MB out for a 32k-token layer of 8 heads.  One launch stands for the torch operations it
// replaced (a comparison with every level, sums, a clone, a fill, a conversion: 110 us of a 32k-token layer, 6 us now), and
// the counts are stored straight into page-locked memory, so that the host waits for one event and no copy.
__global__ __launch_bounds__(LV_THREADS) void finish_levels_kernel(LevelsArgs a) {
    __shared__ int c[12];
    const int row = blockIdx.y, chunk = blockIdx.x, tid = threadIdx.x;
    if (tid < 12) c[tid] = 0;
    __syncthreads();
    int32_t* src = a.bits + (size_t)row * a.T;
    uint8_t* dst = a.levels + (size_t)row * a.stride;
    unsigned long long bulk = 0ull, all = 0ull;
    const int end = min((long long)(chunk + 1) * LV_CHUNK, a.stride);
#pragma unroll
    for (int u = 0; u < LV_CHUNK / (4 * LV_THREADS); ++u) {
        const int t = chunk * LV_CHUNK + (u * LV_THREADS + tid) * 4;
        if (t >= end) continue;
        int b[4] = {16, 16, 16, 16};
        if (a.vec && t + 3 < a.T) {
            const int4 v = *reinterpret_cast<const int4*>(src + t);
            b[0] = v.x; b[1] = v.y; b[2] = v.z; b[3] = v.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) b[e] = t + e < a.T ? src[t + e] : 16;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (t + e >= a.lo && t + e < a.hi) bulk += count_of(b[e]);
            if (t + e >= a.tail && t + e < a.T && b[e] != 16) { b[e] = 16; src[t + e] = 16; }
            if (t + e < a.T) all += count_of(b[e]);
        }
        const uint32_t w = (uint32_t)(b[0] & 0xff) | ((uint32_t)(b[1] & 0xff) << 8) | ((uint32_t)(b[2] & 0xff) << 16) | ((uint32_t)(b[3] & 0xff) << 24);
        *reinterpret_cast<uint32_t*>(dst + t) = w;                    // (stride and base are multiples of four)
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        int x = (int)((bulk >> (6 * k)) & 63ull), y = (int)((all >> (6 * k)) & 63ull);
        int w = x | (y << 16);                                        // both sums stay below 2^16
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) w += __shfl_xor(w, o, WAVE);
        if ((tid & 63) == 0) { atomicAdd(&c[k], w & 0xffff); atomicAdd(&c[6 + k], w >> 16); }
    }
    __syncthreads();
    if (tid < 12) a.counts[((size_t)row * a.chunks + chunk) * 12 + tid] = c[tid];
}

static inline int level_chunks(long long stride) { return (int)((stride + LV_CHUNK - 1) / LV_CHUNK); }

extern "C" int odmkv_finish_levels_chunks(int64_t stride) { return stride > 0 ? level_chunks(stride) : 0; }

extern "C" int odmkv_finish_levels(int32_t* bits, int rows, int T, int count_begin, int count_end, int tail_begin,
                                   uint8_t* levels, int64_t stride, int32_t* counts, void* stream) {
    ODMKV_CHECK_ARG(bits && levels && counts, "finish_levels: null pointer");
    ODMKV_CHECK_ARG(rows > 0 && T > 0, "finish_levels: bad shape rows=%d T=%d", rows, T);
    ODMKV_CHECK_ARG(stride >= T && stride % 4 == 0 && stride < (1ll << 31) && ((uintptr_t)levels & 3) == 0 && ((uintptr_t)bits & 3) == 0,
                    "finish_levels: level rows must hold T tokens and start on multiples of four");
    LevelsArgs a = {bits, levels, counts, (long long)stride, T, count_begin, count_end, tail_begin, level_chunks(stride),
                    (T & 3) == 0 && ((uintptr_t)bits & 15) == 0};
    for (int r0 = 0; r0 < rows; r0 += LV_MAX_ROWS) {                  // (32 layers x 256 sequences x 8 heads are 65536 rows)
        const int n = std::min(rows - r0, LV_MAX_ROWS);
        hipLaunchKernelGGL(finish_levels_kernel, dim3(a.chunks, n), dim3(LV_THREADS), 0, (hipStream_t)stream, a);
        ODMKV_CHECK_LAUNCH("finish_levels_kernel");
        a.bits += (size_t)n * T; a.levels += (size_t)n * stride; a.counts += (size_t)n * a.chunks * 12;
    }
    return 0;
}

// ------------------------------------------------------------------------------------------------
// evicted positions, in the order (sequence, head, token), as three int64 columns
// ------------------------------------------------------------------------------------------------
// (all layers of a prompt in one launch of each kernel: 16 us of latency once, not per layer)
#define EV_LAYERS 64
struct EvictedArgs {
    const uint8_t* levels;
    long long stride;
    int rows, H, T, chunks;              // rows: sequences x heads of a layer
    int32_t* chunk_count;                // [layers, rows, chunks]
    long long* out;                      // per layer [3, n], one behind the other
    long long n[EV_LAYERS];
    long long at[EV_LAYERS];             // element of out where the layer's list starts
};

__device__ static inline int sum256(int v, int* red) {                // over the workgroup, in every thread
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(LV_THREADS) void evicted_count_kernel(EvictedArgs a) {
    __shared__ int red[4];
    const int chunk = blockIdx.x;
    const size_t row = (size_t)blockIdx.z * a.rows + blockIdx.y;
    const uint8_t* src = a.levels + row * a.stride;
    int n = 0;
#pragma unroll
    for (int u = 0; u < LV_CHUNK / LV_THREADS; ++u) {
        const int t = chunk * LV_CHUNK + u * LV_THREADS + threadIdx.x;
        n += t < a.T && src[t] == 0;
    }
    n = sum256(n, red);
    if (threadIdx.x == 0) a.chunk_count[row * a.chunks + chunk] = n;
}

__global__ __launch_bounds__(LV_THREADS) void evicted_list_kernel(EvictedArgs a) {
    __shared__ int red[4];
    const int row = blockIdx.y, layer = blockIdx.z, chunk = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int me = row * a.chunks + chunk;
    const long long total = a.n[layer];
    if (total == 0) return;                                            // (workgroup-uniform)
    const int32_t* counted = a.chunk_count + (size_t)layer * a.rows * a.chunks;
    long long* out = a.out + a.at[layer];
    int before = 0;
    for (int i = tid; i < me; i += LV_THREADS) before += counted[i];
    long long at = sum256(before, red);
    const int b = row / a.H, h = row % a.H;
    const uint8_t* src = a.levels + ((size_t)layer * a.rows + row) * a.stride;
    for (int u = 0; u < LV_CHUNK / LV_THREADS; ++u) {
        const int t = chunk * LV_CHUNK + u * LV_THREADS + tid;
        const bool hit = t < a.T && src[t] == 0;
        const unsigned long long m = __ballot(hit);
        __syncthreads();
        if (lane == 0) red[wave] = __popcll(m);
        __syncthreads();
        int off = __popcll(m & ((1ull << lane) - 1ull));
        for (int w = 0; w < wave; ++w) off += red[w];
        if (hit && at + off < total) {
            out[at + off] = b;
            out[total + at + off] = h;
            out[2 * total + at + off] = t;
        }
        at += red[0] + red[1] + red[2] + red[3];
    }
}

extern "C" size_t odmkv_evicted_layers_workspace_bytes(int layers, int B, int Hkv, int T) {
    return layers > 0 && B > 0 && Hkv > 0 && T > 0 ? (size_t)std::min(layers, EV_LAYERS) * B * Hkv * level_chunks(T) * sizeof(int32_t) : 0;
}

extern "C" int odmkv_evicted_indices_layers(const uint8_t* levels, int layers, int B, int Hkv, int T, int64_t stride, const int64_t* n,
                                     int64_t* out, void* workspace, size_t workspace_bytes, void* stream) {
    ODMKV_CHECK_ARG(levels && n && out && workspace, "evicted_indices: null pointer");
    ODMKV_CHECK_ARG(layers > 0 && B > 0 && Hkv > 0 && T > 0 && (long long)B * Hkv <= 65535 && stride >= T,
                    "evicted_indices: bad shape layers=%d B=%d Hkv=%d T=%d", layers, B, Hkv, T);
    for (int l = 0; l < layers; ++l)
        ODMKV_CHECK_ARG(n[l] >= 0 && n[l] <= (int64_t)B * Hkv * T, "evicted_indices: layer %d cannot hold %lld evicted tokens", l, (long long)n[l]);
    ODMKV_CHECK_ARG(workspace_bytes >= odmkv_evicted_layers_workspace_bytes(layers, B, Hkv, T), "evicted_indices: workspace too small");
    long long at = 0;
    for (int l0 = 0; l0 < layers; l0 += EV_LAYERS) {
        const int m = std::min(layers - l0, EV_LAYERS);
        EvictedArgs a = {levels + (size_t)l0 * B * Hkv * stride, (long long)stride, B * Hkv, Hkv, T, level_chunks(T), (int32_t*)workspace, (long long*)out, {}, {}};
        for (int l = 0; l < m; ++l) { a.n[l] = n[l0 + l]; a.at[l] = at; at += 3 * n[l0 + l]; }
        const dim3 grid(a.chunks, a.rows, m);
        hipLaunchKernelGGL(evicted_count_kernel, grid, dim3(LV_THREADS), 0, (hipStream_t)stream, a);
        ODMKV_CHECK_LAUNCH("evicted_count_kernel");
        hipLaunchKernelGGL(evicted_list_kernel, grid, dim3(LV_THREADS), 0, (hipStream_t)stream, a);
        ODMKV_CHECK_LAUNCH("evicted_list_kernel");
    }
    return 0;
}

extern "C" size_t odmkv_evicted_workspace_bytes(int B, int Hkv, int T) { return odmkv_evicted_layers_workspace_bytes(1, B, Hkv, T); }

extern "C" int odmkv_evicted_indices(const uint8_t* levels, int B, int Hkv, int T, int64_t stride, int64_t n, int64_t* out,
                                     void* workspace, size_t workspace_bytes, void* stream) {
    return odmkv_evicted_indices_layers(levels, 1, B, Hkv, T, stride, &n, out, workspace, workspace_bytes, stream);
}
