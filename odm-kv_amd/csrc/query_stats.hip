// The mean query of a prompt: the mean of the hidden states over the tokens (which the layer's projection then turns into
// the mean query), and the RoPE averaged over the future positions applied to it.
#include <algorithm>
#include "common.h"

#define MN_THREADS 256

// ------------------------------------------------------------------------------------------------
// mean over the rows: x [batch, rows, cols] -> out [batch, cols] of x's type, summed in fp32
// ------------------------------------------------------------------------------------------------
struct MeanArgs {
    const void* x;
    long long sB, sT;                   // elements
    int rows, cols, chunk;              // chunk: rows of a workgroup
    float* part;                        // [batch, chunks, cols]
    void* out;
    int chunks;
};

template <int DT> struct Vec16 { static constexpr int N = DT == ODMKV_F32 ? 4 : 8; };

__device__ static inline uint4 stream16(const void* p) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

template <int DT>
__device__ static inline void add16(const uint4& v, float* acc) {
    if constexpr (DT == ODMKV_F32) {
        acc[0] += __uint_as_float(v.x); acc[1] += __uint_as_float(v.y); acc[2] += __uint_as_float(v.z); acc[3] += __uint_as_float(v.w);
    } else {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[2 * e] += Elem<DT>::to_f32((uint16_t)(w[e] & 0xffffu));
            acc[2 * e + 1] += Elem<DT>::to_f32((uint16_t)(w[e] >> 16));
        }
    }
}

// Bound by HBM: the hidden states once (268 MB for 32k tokens of 4096).  A thread owns 16 bytes of a row and walks its
// workgroup's rows with four requests in flight.  Two workgroups per compute unit with long runs of rows each, and loads that
// leave nothing in the caches, read at 6.4 TB/s (32k x 4096: 42 us; 131k: 159 us, where runs of 256 rows do best); two
// thousand workgroups of 32 rows with plain loads reached 4 TB/s (66 us; 220 us).  The torch form (conversion to fp32, mean)
// moved five times the bytes: 250 us.  The sums are formed in another order than torch's; rounded to 16 bits, 0 to 3 columns in
// 10000 are not the nearest value to the fp64 mean (300 to 131072 tokens; torch's fp32 mean 0 to 5), so that a mean query may land
// one step of its type apart from torch's.
template <int DT>
__global__ __launch_bounds__(MN_THREADS) void mean_part_kernel(MeanArgs a) {
    constexpr int N = Vec16<DT>::N, U = 4;
    const int col = (blockIdx.x * MN_THREADS + threadIdx.x) * N;
    if (col >= a.cols) return;                                        // (cols is a multiple of N)
    const int r0 = blockIdx.y * a.chunk, r1 = min(r0 + a.chunk, a.rows);
    constexpr int BYTES = DT == ODMKV_F32 ? 4 : 2;
    const char* p = (const char*)a.x + ((long long)blockIdx.z * a.sB + (long long)r0 * a.sT + col) * BYTES;
    const long long step = a.sT * BYTES;
    float acc[N];
#pragma unroll
    for (int e = 0; e < N; ++e) acc[e] = 0.0f;
    int r = r0;
    for (; r + U <= r1; r += U) {
        uint4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = stream16(p + u * step);
        p += U * step;
#pragma unroll
        for (int u = 0; u < U; ++u) add16<DT>(v[u], acc);
    }
    for (; r < r1; ++r, p += step) add16<DT>(*reinterpret_cast<const uint4*>(p), acc);
    float* o = a.part + ((size_t)blockIdx.z * a.chunks + blockIdx.y) * a.cols + col;
#pragma unroll
    for (int e = 0; e < N; e += 4) *reinterpret_cast<float4*>(o + e) = make_float4(acc[e], acc[e + 1], acc[e + 2], acc[e + 3]);
}

// sixteen columns and sixteen shares of the chunks per workgroup
template <int DT>
__global__ __launch_bounds__(MN_THREADS) void mean_final_kernel(MeanArgs a) {
    __shared__ float red[16][17];
    const int c = threadIdx.x & 15, g = threadIdx.x >> 4, col = blockIdx.x * 16 + c;
    float s = 0.0f;
    if (col < a.cols) {
        const float* p = a.part + (size_t)blockIdx.z * a.chunks * a.cols + col;
#pragma unroll 8
        for (int k = g; k < a.chunks; k += 16) s += p[(size_t)k * a.cols];
    }
    red[g][c] = s;
    __syncthreads();
    if (g == 0 && col < a.cols) {
        float t = 0.0f;
#pragma unroll
        for (int k = 0; k < 16; ++k) t += red[k][c];
        reinterpret_cast<typename Elem<DT>::raw*>(a.out)[(size_t)blockIdx.z * a.cols + col] = Elem<DT>::from_f32(t / (float)a.rows);
    }
}

// row runs that put two workgroups on every compute unit
static int mean_runs(int batch, int cols, int per_thread) {
    const long long blocks = ((cols + MN_THREADS * per_thread - 1) / (MN_THREADS * per_thread)) * (long long)batch;
    return (int)std::max<long long>(1, 512 / blocks);
}
#define MN_CHUNK_MIN 16
#define MN_CHUNK_MAX 256
static int mean_chunk(int batch, int rows, int cols, int per_thread) {
    const int runs = mean_runs(batch, cols, per_thread);
    return std::min(MN_CHUNK_MAX, std::max(MN_CHUNK_MIN, (int)(((long long)rows + runs - 1) / runs)));
}

// Room for the partial sums of any call with at most `rows` rows.  (The parts of one call, ceil(rows / chunk), are no monotone
// function of its rows: 8193 rows in runs of 33 make 249, 8189 in runs of 32 make 256.)
extern "C" size_t odmkv_token_mean_workspace_bytes(int batch, int rows, int cols) {
    if (batch <= 0 || rows <= 0 || cols <= 0) return 0;
    const long long runs = std::max(mean_runs(batch, cols, 8), mean_runs(batch, cols, 4));
    const long long shortest = ((long long)rows + MN_CHUNK_MIN - 1) / MN_CHUNK_MIN, longest = ((long long)rows + MN_CHUNK_MAX - 1) / MN_CHUNK_MAX;
    return (size_t)batch * std::min(shortest, std::max(runs, longest)) * cols * sizeof(float);
}

extern "C" int odmkv_token_mean(const void* x, int dtype, int batch, int rows, int cols, int64_t stride_b, int64_t stride_t,
                                void* out, void* workspace, size_t workspace_bytes, void* stream) {
    ODMKV_CHECK_ARG(x && out && workspace, "token_mean: null pointer");
    ODMKV_CHECK_ARG(dtype == ODMKV_F16 || dtype == ODMKV_BF16 || dtype == ODMKV_F32, "token_mean: bad dtype %d", dtype);
    ODMKV_CHECK_ARG(batch > 0 && batch <= 65535 && rows > 0 && cols > 0, "token_mean: bad shape batch=%d rows=%d cols=%d", batch, rows, cols);
    const int n = dtype == ODMKV_F32 ? 4 : 8;
    ODMKV_CHECK_ARG(cols % n == 0 && stride_b % n == 0 && stride_t % n == 0 && ((uintptr_t)x & 15) == 0,
                    "token_mean: rows must start on multiples of 16 bytes and hold whole ones");
    ODMKV_CHECK_ARG(workspace_bytes >= odmkv_token_mean_workspace_bytes(batch, rows, cols), "token_mean: workspace too small");
    MeanArgs a = {x, (long long)stride_b, (long long)stride_t, rows, cols, mean_chunk(batch, rows, cols, n), (float*)workspace, out, 0};
    a.chunks = (rows + a.chunk - 1) / a.chunk;
    const dim3 grid((cols / n + MN_THREADS - 1) / MN_THREADS, a.chunks, batch), final_grid((cols + 15) / 16, 1, batch);
    hipStream_t st = (hipStream_t)stream;
#define MEAN_LAUNCH(DT)                                                                         \
    hipLaunchKernelGGL(mean_part_kernel<DT>, grid, dim3(MN_THREADS), 0, st, a);                  \
    hipLaunchKernelGGL(mean_final_kernel<DT>, final_grid, dim3(MN_THREADS), 0, st, a)
    if (dtype == ODMKV_F16) { MEAN_LAUNCH(ODMKV_F16); }
    else if (dtype == ODMKV_BF16) { MEAN_LAUNCH(ODMKV_BF16); }
    else { MEAN_LAUNCH(ODMKV_F32); }
#undef MEAN_LAUNCH
    ODMKV_CHECK_LAUNCH("mean_part_kernel");
    return 0;
}

// ------------------------------------------------------------------------------------------------
// projection of a few rows: out[b][r] = sum_c w[r][c] x[b][c] + bias[r], summed in fp32, rounded to w's type
// ------------------------------------------------------------------------------------------------
struct ProjectArgs {
    const uint16_t* w;                  // [rows, cols], ld elements apart
    const uint16_t* bias;               // [rows] or null
    const uint16_t* x;                  // [NB, cols]
    long long ld;
    int rows, cols;
    void* out;                          // [NB, rows] of w's type, or those values widened to fp32
    int wide;
};

// Bound by HBM: the weight once (33 MB for 4096 x 4096).  A wavefront takes two rows with eight requests in flight, so that
// 4096 rows put 2048 wavefronts on the device: 9 us against 13 us for the library's product with one row, and a quarter of
// the host's time.
template <int DT, int NB>
__global__ __launch_bounds__(MN_THREADS) void project_rows_kernel(ProjectArgs a) {
    constexpr int U = 4;
    const int lane = threadIdx.x & 63, r0 = (blockIdx.x * (MN_THREADS / 64) + (threadIdx.x >> 6)) * 2;
    if (r0 >= a.rows) return;
    const int r1 = min(r0 + 1, a.rows - 1);
    float acc[NB][2];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b][0] = acc[b][1] = 0.0f;
    auto dot8 = [](const uint4& u, const uint4& v, float s) {
        const uint32_t p[4] = {u.x, u.y, u.z, u.w}, q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s = __fmaf_rn(Elem<DT>::to_f32((uint16_t)(p[e] & 0xffffu)), Elem<DT>::to_f32((uint16_t)(q[e] & 0xffffu)), s);
            s = __fmaf_rn(Elem<DT>::to_f32((uint16_t)(p[e] >> 16)), Elem<DT>::to_f32((uint16_t)(q[e] >> 16)), s);
        }
        return s;
    };
    for (int c0 = 0; c0 < a.cols; c0 += U * 512) {
        uint4 w0[U], w1[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = c0 + u * 512 + lane * 8;
            w0[u] = w1[u] = make_uint4(0u, 0u, 0u, 0u);
            if (c < a.cols) {                                            // (cols is a multiple of eight)
                w0[u] = *reinterpret_cast<const uint4*>(a.w + r0 * a.ld + c);
                w1[u] = *reinterpret_cast<const uint4*>(a.w + r1 * a.ld + c);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int c = c0 + u * 512 + lane * 8;
            if (c >= a.cols) continue;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const uint4 x = *reinterpret_cast<const uint4*>(a.x + (size_t)b * a.cols + c);
                acc[b][0] = dot8(w0[u], x, acc[b][0]);
                acc[b][1] = dot8(w1[u], x, acc[b][1]);
            }
        }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const float t = wave_sum(acc[b][k]);
            const int r = r0 + k;
            if (lane == 0 && r < a.rows) {
                const uint16_t v = Elem<DT>::from_f32(a.bias ? t + Elem<DT>::to_f32(a.bias[r]) : t);
                const size_t at = (size_t)b * a.rows + r;
                if (a.wide) reinterpret_cast<float*>(a.out)[at] = Elem<DT>::to_f32(v);
                else reinterpret_cast<uint16_t*>(a.out)[at] = v;
            }
        }
}

extern "C" int odmkv_project_rows(const void* weight, int64_t ld, const void* bias, const void* x, int dtype, int batch, int rows,
                                  int cols, void* out, int out_dtype, void* stream) {
    ODMKV_CHECK_ARG(weight && x && out, "project_rows: null pointer");
    ODMKV_CHECK_ARG((dtype == ODMKV_F16 || dtype == ODMKV_BF16) && (out_dtype == dtype || out_dtype == ODMKV_F32), "project_rows: bad dtype %d -> %d", dtype, out_dtype);
    ODMKV_CHECK_ARG(batch > 0 && rows > 0 && cols > 0 && cols % 8 == 0 && ld >= cols && ld % 8 == 0 && (((uintptr_t)weight | (uintptr_t)x) & 15) == 0,
                    "project_rows: rows must start on multiples of 16 bytes and hold whole ones (rows=%d cols=%d)", rows, cols);
    const dim3 grid((rows + 2 * (MN_THREADS / 64) - 1) / (2 * (MN_THREADS / 64))), block(MN_THREADS);
    hipStream_t st = (hipStream_t)stream;
    const size_t wide = out_dtype == ODMKV_F32 ? 4 : 2;
    for (int b = 0; b < batch;) {                                         // (up to four rows share a pass over the weight)
        const int n = batch - b >= 4 ? 4 : batch - b >= 2 ? 2 : 1;
        const ProjectArgs a = {(const uint16_t*)weight, (const uint16_t*)bias, (const uint16_t*)x + (size_t)b * cols, (long long)ld, rows, cols,
                               (char*)out + (size_t)b * rows * wide, out_dtype == ODMKV_F32};
#define PROJECT(DT)                                                                             \
        if (n == 4) hipLaunchKernelGGL((project_rows_kernel<DT, 4>), grid, block, 0, st, a);     \
        else if (n == 2) hipLaunchKernelGGL((project_rows_kernel<DT, 2>), grid, block, 0, st, a); \
        else hipLaunchKernelGGL((project_rows_kernel<DT, 1>), grid, block, 0, st, a)
        if (dtype == ODMKV_F16) { PROJECT(ODMKV_F16); } else { PROJECT(ODMKV_BF16); }
#undef PROJECT
        ODMKV_CHECK_LAUNCH("project_rows_kernel");
        b += n;
    }
    return 0;
}

// ------------------------------------------------------------------------------------------------
// averaged RoPE: out = c * mu + s * rotate_half(mu), c and s the means of cos and sin over the positions, every step
// rounded to the tensors' type as the tensor operations it stands for do; the result widened to fp32
// ------------------------------------------------------------------------------------------------
struct RopeArgs {
    const void* mu;                     // [heads, 128]
    const void* cosine;                 // [positions, 128]
    const void* sine;
    int heads, positions;
    float* out;                         // [heads, 128]
};

// Bound by latency (128 KB of tables out of the L2 for 512 positions).  A workgroup takes sixteen columns; one launch for
// eight: 45 us of kernels and as much host time per layer before, 5 us now.
template <int DT>
__global__ __launch_bounds__(MN_THREADS) void average_rope_kernel(RopeArgs a) {
    __shared__ float red_c[16][17], red_s[16][17];
    __shared__ float c_bar[16], s_bar[16];
    typedef typename Elem<DT>::raw raw;
    auto round_dt = [](float x) { return Elem<DT>::to_f32(Elem<DT>::from_f32(x)); };
    const int c = threadIdx.x & 15, g = threadIdx.x >> 4, col = blockIdx.x * 16 + c;
    float sc = 0.0f, ss = 0.0f;
#pragma unroll 8
    for (int p = g; p < a.positions; p += 16) {
        sc += Elem<DT>::to_f32(reinterpret_cast<const raw*>(a.cosine)[(size_t)p * HD + col]);
        ss += Elem<DT>::to_f32(reinterpret_cast<const raw*>(a.sine)[(size_t)p * HD + col]);
    }
    red_c[g][c] = sc; red_s[g][c] = ss;
    __syncthreads();
    if (g < 2) {
        float t = 0.0f;
#pragma unroll
        for (int k = 0; k < 16; ++k) t += g == 0 ? red_c[k][c] : red_s[k][c];
        (g == 0 ? c_bar : s_bar)[c] = round_dt(t / (float)a.positions);
    }
    __syncthreads();
    for (int h = g; h < a.heads; h += 16) {
        const raw* row = reinterpret_cast<const raw*>(a.mu) + (size_t)h * HD;
        const float x = Elem<DT>::to_f32(row[col]), o = Elem<DT>::to_f32(row[col ^ 64]);
        const float rot = col < 64 ? -o : o;
        a.out[(size_t)h * HD + col] = round_dt(round_dt(c_bar[c] * x) + round_dt(s_bar[c] * rot));
    }
}

extern "C" int odmkv_average_rope(const void* mu, const void* cosine, const void* sine, int dtype, int heads, int positions,
                                  float* out, void* stream) {
    ODMKV_CHECK_ARG(mu && cosine && sine && out, "average_rope: null pointer");
    ODMKV_CHECK_ARG(dtype == ODMKV_F16 || dtype == ODMKV_BF16 || dtype == ODMKV_F32, "average_rope: bad dtype %d", dtype);
    ODMKV_CHECK_ARG(heads > 0 && positions > 0, "average_rope: bad shape heads=%d positions=%d", heads, positions);
    const RopeArgs a = {mu, cosine, sine, heads, positions, out};
    const dim3 grid(HD / 16), block(MN_THREADS);
    hipStream_t st = (hipStream_t)stream;
    if (dtype == ODMKV_F16) hipLaunchKernelGGL(average_rope_kernel<ODMKV_F16>, grid, block, 0, st, a);
    else if (dtype == ODMKV_BF16) hipLaunchKernelGGL(average_rope_kernel<ODMKV_BF16>, grid, block, 0, st, a);
    else hipLaunchKernelGGL(average_rope_kernel<ODMKV_F32>, grid, block, 0, st, a);
    ODMKV_CHECK_LAUNCH("average_rope_kernel");
    return 0;
}

// ------------------------------------------------------------------------------------------------
// mean and covariance of the queries of every head, passed through the averaged RoPE:
//   mu = sum_t q_t / n,  C = sum_t (q_t - mu) (q_t - mu)^T / n,  mu' = R mu,  C' = R C R^T,  R = diag(c) + diag(s) (half rotation)
// The queries are taken relative to a pivot near their mean (the mean of 64 of them, the same for every workgroup of a head),
// x = q - pivot in fp32, and x as three bf16 pieces whose sum it is: six products of pieces on the matrix cores (what they
// leave out, second times third piece twice and third times third, is up to 2^-21 of the product, always with its sign, where x
// has all of fp32's bits), fp32 sums over at most 512 tokens at a time, fp64 behind that, where the rest of the mean is
// subtracted.  The pivot is rounded to the queries' type: q - pivot and its running sum then mostly are exact, and the third
// piece is mostly empty.  (With all of fp32's bits in the pivot every addition to a running sum was off by the same share of
// its last place.)  Off fp64 over 600 to 32768 tokens, relative: means through the RoPE 0.3e-7 to 0.5e-7 (with such a pivot
// 1.0e-7 to 5.1e-7; tensor operations in fp32 0.6e-7 to 1.2e-7), covariances 0.7e-7 to 1.7e-7 (1.2e-7 to 4.5e-7; 3.9e-7 to 2.7e-6).
// (Products of the 16-bit queries as they are would be exact and a sixth of the work, but with a mean several
// times the deviation their fp32 sums keep less of the covariance than sums of centred queries do.)
// v_mfma_f32_32x32x16_bf16: D[32x32] += A[32x16] B[16x32], lane l supplies A[l % 32][8 (l / 32) + e] and the same of B^T:
// both operands are the queries with the dims along the lanes and eight tokens in a lane.  A lane loads four dims
// (4 p .. 4 p + 3, p = l % 32) of eight tokens and pairs the tokens up by byte permutes: block b = the dims 4 p + b.  Ten of the
// sixteen 32x32 blocks (the others mirror them).
// Floors for 32 heads of 32k tokens: 268 MB once, 129 GFLOP of bf16 products.  As tensor operations (conversion, mean,
// subtraction, fp32 product) 1050 us, here 139 + 15 (bound by the matrix cores: 0.93 PFLOP/s).
// ------------------------------------------------------------------------------------------------
#define CV_WAVES 8
#define CV_BLOCKS 10                 // (0,0) (0,1) (0,2) (0,3) (1,1) (1,2) (1,3) (2,2) (2,3) (3,3)
#define CV_PART (CV_BLOCKS * 1024 + 2 * HD)      // blocks, sum of x, pivot
#define CV_TOKENS 512                // tokens a wavefront sums in fp32
#define CV_SAMPLE 64                 // tokens of the pivot
typedef float cv_f16 __attribute__((ext_vector_type(16)));
typedef __bf16 cv_b8 __attribute__((ext_vector_type(8)));

__device__ static __forceinline__ cv_f16 cv_mfma(const uint4& a, const uint4& b, const cv_f16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(cv_b8, a), __builtin_bit_cast(cv_b8, b), c, 0, 0, 0);
}

struct CovArgs {
    const uint16_t* q;                   // head h, token t at h * sH + t * sT
    long long sH, sT;
    int tokens, slices, per_wave;        // per_wave: a multiple of 16
    float* part;                         // [heads, slices, CV_PART]
    const float* cosine;                 // [positions, 128] or null: no RoPE
    const float* sine;
    int positions;
    float* rope;                         // [2, 128]
    float* mu;                           // [heads, 128]
    float* cov;                          // [heads, 128, 128]
};

template <int DT>
__global__ __launch_bounds__(CV_WAVES * 64) void cov_part_kernel(CovArgs a) {
    __shared__ float red[2][CV_WAVES][1024];
    __shared__ float sums[CV_WAVES][HD];
    __shared__ __align__(16) float pivot[HD];
    const int slice = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = lane & 31, half = lane >> 5;
    const int t0 = (slice * CV_WAVES + wave) * a.per_wave, t1 = min(t0 + a.per_wave, a.tokens);
    const uint16_t* head = a.q + (long long)h * a.sH;
    const uint16_t* base = head + 4 * p;
    uint2 cur[8];
    const auto request = [&](int t) {
#pragma unroll
        for (int e = 0; e < 8; ++e) cur[e] = *reinterpret_cast<const uint2*>(base + (long long)min(t + 8 * half + e, a.tokens - 1) * a.sT);
    };
    {
        float s = 0.0f;
        uint16_t v[CV_SAMPLE / 4];
#pragma unroll
        for (int i = 0; i < CV_SAMPLE / 4; ++i)
            v[i] = head[(long long)(((long long)(4 * i + (tid >> 7)) * a.tokens) / CV_SAMPLE) * a.sT + (tid & 127)];
        if (t0 < t1) request(t0);
#pragma unroll
        for (int i = 0; i < CV_SAMPLE / 4; ++i) s += Elem<DT>::to_f32(v[i]);
        sums[tid >> 7][tid & 127] = s;
        __syncthreads();
        if (tid < HD) pivot[tid] = Elem<DT>::to_f32(Elem<DT>::from_f32((sums[0][tid] + sums[1][tid] + sums[2][tid] + sums[3][tid]) / (float)CV_SAMPLE));
        __syncthreads();
    }
    const float4 c4 = *reinterpret_cast<const float4*>(pivot + 4 * p);
    const float c[4] = {c4.x, c4.y, c4.z, c4.w};
    cv_f16 acc[CV_BLOCKS];
#pragma unroll
    for (int b = 0; b < CV_BLOCKS; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[b][r] = 0.0f;
    float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int t = t0; t < t1; t += 16) {
        uint4 op[3][4];                                               // pieces of the four blocks
        const bool ragged = t + 16 > t1;                              // the last step (wave-uniform)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            uint32_t w[3][4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float x[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint32_t two = b < 2 ? cur[2 * r + k].x : cur[2 * r + k].y;
                    x[k] = Elem<DT>::to_f32((uint16_t)((b & 1) ? two >> 16 : two & 0xffffu)) - c[b];
                    if (ragged && t + 8 * half + 2 * r + k >= t1) x[k] = 0.0f;
                    sum[b] += x[k];
                }
#pragma unroll
                for (int i = 0; i < 3; ++i) {                         // the upper half of each as a bf16 piece; the rest stays
                    const uint32_t u0 = __float_as_uint(x[0]), u1 = __float_as_uint(x[1]);
                    w[i][r] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
                    x[0] -= __uint_as_float(u0 & 0xffff0000u);
                    x[1] -= __uint_as_float(u1 & 0xffff0000u);
                }
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) op[i][b] = make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]);
        }
        if (t + 16 < t1) request(t + 16);                             // on their way under the products
        int k = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = i; j < 4; ++j, ++k) {                        // small pieces first
                acc[k] = cv_mfma(op[2][i], op[0][j], acc[k]);
                acc[k] = cv_mfma(op[0][i], op[2][j], acc[k]);
                acc[k] = cv_mfma(op[1][i], op[1][j], acc[k]);
                acc[k] = cv_mfma(op[1][i], op[0][j], acc[k]);
                acc[k] = cv_mfma(op[0][i], op[1][j], acc[k]);
                acc[k] = cv_mfma(op[0][i], op[0][j], acc[k]);
            }
    }
    __syncthreads();                                                  // (the sums' space held the pivot's shares)
    // the eight wavefronts' blocks added up, one block at a time
    float* part = a.part + ((size_t)h * a.slices + slice) * CV_PART;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const float s = sum[b] + __shfl_xor(sum[b], 32, WAVE);
        if (half == 0) sums[wave][4 * p + b] = s;
    }
#pragma unroll
    for (int k = 0; k < CV_BLOCKS; ++k) {
#pragma unroll
        for (int r = 0; r < 16; ++r) red[k & 1][wave][r * 64 + lane] = acc[k][r];
        __syncthreads();
#pragma unroll
        for (int e = tid; e < 1024; e += CV_WAVES * 64) {
            float s = 0.0f;
#pragma unroll
            for (int w = 0; w < CV_WAVES; ++w) s += red[k & 1][w][e];
            part[k * 1024 + e] = s;
        }
    }
    if (tid < HD) {
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < CV_WAVES; ++w) s += sums[w][tid];
        part[CV_BLOCKS * 1024 + tid] = s;
        part[CV_BLOCKS * 1024 + HD + tid] = pivot[tid];
    }
}

// means of cos and sin over the positions (a workgroup per sixteen columns)
__global__ __launch_bounds__(MN_THREADS) void rope_mean_kernel(CovArgs a) {
    __shared__ double red[2][16][17];
    const int c = threadIdx.x & 15, g = threadIdx.x >> 4, col = blockIdx.x * 16 + c;
    double sc = 0.0, ss = 0.0;                                        // (cos and sin cancel over the positions)
#pragma unroll 8
    for (int x = g; x < a.positions; x += 16) { sc += a.cosine[(size_t)x * HD + col]; ss += a.sine[(size_t)x * HD + col]; }
    red[0][g][c] = sc; red[1][g][c] = ss;
    __syncthreads();
    if (g < 2) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) t += red[g][k][c];
        a.rope[g * HD + col] = (float)(t / a.positions);
    }
}

// element (i, j) of the sum of q q^T: which block, and where D of a 32x32 matrix instruction keeps it (lane = 32 (x / 4 % 2) + column,
// register 4 (x / 8) + x % 4 of row x)
__device__ static inline int cov_at(int i, int j) {
    int bi = i & 3, bj = j & 3, x = i >> 2, y = j >> 2;
    if (bi > bj || (bi == bj && x > y)) { const int t = bi; bi = bj; bj = t; const int u = x; x = y; y = u; }
    const int k = bi * 4 - bi * (bi - 1) / 2 + (bj - bi);
    return k * 1024 + (4 * (x >> 3) + (x & 3)) * 64 + 32 * ((x >> 2) & 1) + y;
}

// A workgroup: rows i and i + 64 of four i < 64 of one head
__global__ __launch_bounds__(256) void cov_final_kernel(CovArgs a) {
    __shared__ double mean[HD];
    __shared__ float c[8][HD];
    __shared__ float cs[2][HD];
    const int h = blockIdx.y, tid = threadIdx.x;
    const float* part = a.part + (size_t)h * a.slices * CV_PART;
    // A thread's four entries and its share of the means, eight slices of each asked for at once (one after the other they were a chain
    // of forty round trips: 26 us a call of 32 heads of 32k tokens, 15 now); added up in the slices' order
    double s[4] = {0.0, 0.0, 0.0, 0.0}, sm = 0.0;
    int at[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = tid + 256 * u, r = e >> 7;
        at[u] = cov_at(blockIdx.x * 4 + (r & 3) + 64 * (r >> 2), e & 127);
    }
    for (int k0 = 0; k0 < a.slices; k0 += 8) {
        float v[4][8], vm[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float* slice = part + (size_t)min(k0 + k, a.slices - 1) * CV_PART;
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u][k] = slice[at[u]];
            vm[k] = slice[CV_BLOCKS * 1024 + (tid & (HD - 1))];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (k0 + k >= a.slices) break;
#pragma unroll
            for (int u = 0; u < 4; ++u) s[u] += (double)v[u][k];
            sm += (double)vm[k];
        }
    }
    if (tid < HD) {
        mean[tid] = sm / a.tokens;                           // relative to the pivot
        cs[0][tid] = a.cosine ? a.rope[tid] : 1.0f;
        cs[1][tid] = a.cosine ? a.rope[HD + tid] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = tid + 256 * u, r = e >> 7, i = blockIdx.x * 4 + (r & 3) + 64 * (r >> 2), j = e & 127;
        c[r][j] = (float)(s[u] / a.tokens - mean[i] * mean[j]);
    }
    __syncthreads();
    for (int e = tid; e < 8 * HD; e += 256) {
        const int r = e >> 7, i = blockIdx.x * 4 + (r & 3) + 64 * (r >> 2), j = e & 127;
        const float rj = j < 64 ? -1.0f : 1.0f, ri = i < 64 ? -1.0f : 1.0f;
        // the map on the last axis of rows i and i +- 64, then across them
        const float own = cs[0][j] * c[r][j] + cs[1][j] * (rj * c[r][j ^ 64]);
        const float other = cs[0][j] * c[r ^ 4][j] + cs[1][j] * (rj * c[r ^ 4][j ^ 64]);
        a.cov[((size_t)h * HD + i) * HD + j] = cs[0][i] * own + cs[1][i] * (ri * other);
    }
    if (blockIdx.x == 0 && tid < HD) {
        const float* pivot = part + CV_BLOCKS * 1024 + HD;
        const double m = mean[tid] + pivot[tid], o = mean[tid ^ 64] + pivot[tid ^ 64];
        a.mu[(size_t)h * HD + tid] = (float)(cs[0][tid] * m + cs[1][tid] * (tid < 64 ? -o : o));
    }
}

static int cov_slices(int tokens) { return std::max(8, (tokens + CV_WAVES * CV_TOKENS - 1) / (CV_WAVES * CV_TOKENS)); }

extern "C" size_t odmkv_query_covariance_workspace_bytes(int heads, int tokens) {
    return heads > 0 && tokens > 0 ? ((size_t)heads * cov_slices(tokens) * CV_PART + 2 * HD) * sizeof(float) : 0;
}

extern "C" int odmkv_query_covariance(const void* q, int dtype, int heads, int tokens, int64_t stride_h, int64_t stride_t,
                                      const float* cosine, const float* sine, int positions, float* mu, float* cov,
                                      void* workspace, size_t workspace_bytes, void* stream) {
    ODMKV_CHECK_ARG(q && mu && cov && workspace, "query_covariance: null pointer");
    ODMKV_CHECK_ARG(dtype == ODMKV_F16 || dtype == ODMKV_BF16, "query_covariance: 16-bit queries only");
    ODMKV_CHECK_ARG(heads > 0 && heads <= 65535 && tokens > 0, "query_covariance: bad shape heads=%d tokens=%d", heads, tokens);
    ODMKV_CHECK_ARG((cosine == nullptr) == (sine == nullptr) && (!cosine || positions > 0), "query_covariance: bad RoPE tables");
    ODMKV_CHECK_ARG(((uintptr_t)q & 7) == 0 && stride_h % 4 == 0 && stride_t % 4 == 0, "query_covariance: rows must start on multiples of 8 bytes");
    ODMKV_CHECK_ARG(workspace_bytes >= odmkv_query_covariance_workspace_bytes(heads, tokens), "query_covariance: workspace too small");
    CovArgs a;
    a.q = (const uint16_t*)q; a.sH = stride_h; a.sT = stride_t; a.tokens = tokens;
    a.slices = cov_slices(tokens);
    a.per_wave = ((tokens + a.slices * CV_WAVES - 1) / (a.slices * CV_WAVES) + 15) & ~15;
    a.part = (float*)workspace; a.rope = a.part + (size_t)heads * a.slices * CV_PART;
    a.cosine = cosine; a.sine = sine; a.positions = positions; a.mu = mu; a.cov = cov;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == ODMKV_F16) hipLaunchKernelGGL(cov_part_kernel<ODMKV_F16>, dim3(a.slices, heads), dim3(CV_WAVES * 64), 0, st, a);
    else hipLaunchKernelGGL(cov_part_kernel<ODMKV_BF16>, dim3(a.slices, heads), dim3(CV_WAVES * 64), 0, st, a);
    ODMKV_CHECK_LAUNCH("cov_part_kernel");
    if (cosine) {
        hipLaunchKernelGGL(rope_mean_kernel, dim3(HD / 16), dim3(MN_THREADS), 0, st, a);
        ODMKV_CHECK_LAUNCH("rope_mean_kernel");
    }
    hipLaunchKernelGGL(cov_final_kernel, dim3(16, heads), dim3(256), 0, st, a);
    ODMKV_CHECK_LAUNCH("cov_final_kernel");
    return 0;
}

// ------------------------------------------------------------------------------------------------
// RoPE of a window's queries: q [heads, tokens, 128] with strides -> contiguous, q * cos + rotate_half(q) * sin with every
// product and the sum rounded to the type (one launch for six)
// ------------------------------------------------------------------------------------------------
struct RotateArgs { const void* q; long long sH, sT; const void* cosine; const void* sine; int heads, tokens; void* out; };

template <int DT>
__global__ __launch_bounds__(256) void rotate_queries_kernel(RotateArgs a) {
    typedef typename Elem<DT>::raw raw;
    auto round_dt = [](float x) { return Elem<DT>::to_f32(Elem<DT>::from_f32(x)); };
    const int i = blockIdx.x * 256 + threadIdx.x, col = i & 127, row = i >> 7;
    if (row >= a.heads * a.tokens) return;
    const int t = row % a.tokens;
    const raw* src = (const raw*)a.q + (long long)(row / a.tokens) * a.sH + (long long)t * a.sT;
    const float x = Elem<DT>::to_f32(src[col]), o = Elem<DT>::to_f32(src[col ^ 64]);
    const float c = Elem<DT>::to_f32(((const raw*)a.cosine)[t * HD + col]), s = Elem<DT>::to_f32(((const raw*)a.sine)[t * HD + col]);
    ((raw*)a.out)[i] = Elem<DT>::from_f32(round_dt(x * c) + round_dt((col < 64 ? -o : o) * s));
}

extern "C" int odmkv_rotate_queries(const void* q, int dtype, int heads, int tokens, int64_t stride_h, int64_t stride_t,
                                    const void* cosine, const void* sine, void* out, void* stream) {
    ODMKV_CHECK_ARG(q && cosine && sine && out, "rotate_queries: null pointer");
    ODMKV_CHECK_ARG(dtype == ODMKV_F16 || dtype == ODMKV_BF16 || dtype == ODMKV_F32, "rotate_queries: bad dtype %d", dtype);
    ODMKV_CHECK_ARG(heads > 0 && tokens > 0 && (long long)heads * tokens < (1ll << 24), "rotate_queries: bad shape heads=%d tokens=%d", heads, tokens);
    const RotateArgs a = {q, (long long)stride_h, (long long)stride_t, cosine, sine, heads, tokens, out};
    const dim3 grid((heads * tokens * HD + 255) / 256), block(256);
    hipStream_t st = (hipStream_t)stream;
    if (dtype == ODMKV_F16) hipLaunchKernelGGL(rotate_queries_kernel<ODMKV_F16>, grid, block, 0, st, a);
    else if (dtype == ODMKV_BF16) hipLaunchKernelGGL(rotate_queries_kernel<ODMKV_BF16>, grid, block, 0, st, a);
    else hipLaunchKernelGGL(rotate_queries_kernel<ODMKV_F32>, grid, block, 0, st, a);
    ODMKV_CHECK_LAUNCH("rotate_queries_kernel");
    return 0;
}

// ------------------------------------------------------------------------------------------------
// scores in [0, 1] over the whole layer: (x - lo) / (hi - lo), one half everywhere where hi - lo < 1e-8; pad > 0: the rows get
// that many columns of the largest score in front (the sinks).  The decision stays on the device (as tensor operations the
// host waited for it), two launches for six.
// ------------------------------------------------------------------------------------------------
#define NRM_GROUPS 256
struct NormalizeArgs { const float* x; long long rows, cols; int pad, scale; float* part; float* out; };

// torch's amin / amax: a NaN anywhere is the result
__device__ static inline float nan_min(float a, float b) { return a != a || b != b ? NAN : fminf(a, b); }
__device__ static inline float nan_max(float a, float b) { return a != a || b != b ? NAN : fmaxf(a, b); }
__device__ static inline void wg_minmax(float& lo, float& hi, float (*red)[2]) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { lo = nan_min(lo, __shfl_xor(lo, o, WAVE)); hi = nan_max(hi, __shfl_xor(hi, o, WAVE)); }
    if ((threadIdx.x & 63) == 0) { red[threadIdx.x >> 6][0] = lo; red[threadIdx.x >> 6][1] = hi; }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 4; ++w) { lo = nan_min(lo, red[w][0]); hi = nan_max(hi, red[w][1]); }
}

__global__ __launch_bounds__(256) void minmax_kernel(NormalizeArgs a) {
    __shared__ float red[4][2];
    const long long n = a.rows * a.cols, step = (long long)gridDim.x * 256;
    float lo = INFINITY, hi = -INFINITY;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += step) { const float v = a.x[i]; lo = nan_min(lo, v); hi = nan_max(hi, v); }
    wg_minmax(lo, hi, red);
    if (threadIdx.x == 0) { a.part[2 * blockIdx.x] = lo; a.part[2 * blockIdx.x + 1] = hi; }
}

__global__ __launch_bounds__(256) void normalize_kernel(NormalizeArgs a) {
    __shared__ float red[4][2];
    float lo = a.part[2 * threadIdx.x], hi = a.part[2 * threadIdx.x + 1];
    wg_minmax(lo, hi, red);
    const float span = hi - lo;
    const bool flat = span < 1e-8f;
    const long long cols = a.cols + a.pad, n = a.rows * cols, step = (long long)gridDim.x * 256;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
        const long long r = i / cols, c = i - r * cols;
        const float v = c < a.pad ? hi : a.x[r * a.cols + c - a.pad];
        a.out[i] = !a.scale ? v : flat ? 0.5f : (v - lo) / span;
    }
}

extern "C" size_t odmkv_normalize_workspace_bytes(void) { return NRM_GROUPS * 2 * sizeof(float); }

extern "C" int odmkv_normalize_scores(const float* scores, int64_t rows, int64_t cols, int pad, int scale, float* out,
                                      void* workspace, size_t workspace_bytes, void* stream) {
    ODMKV_CHECK_ARG(scores && out && workspace, "normalize_scores: null pointer");
    ODMKV_CHECK_ARG(rows > 0 && cols > 0 && pad >= 0, "normalize_scores: bad shape");
    ODMKV_CHECK_ARG(workspace_bytes >= odmkv_normalize_workspace_bytes(), "normalize_scores: workspace too small");
    const NormalizeArgs a = {scores, (long long)rows, (long long)cols, pad, scale, (float*)workspace, out};
    hipLaunchKernelGGL(minmax_kernel, dim3(NRM_GROUPS), dim3(256), 0, (hipStream_t)stream, a);
    const long long n = (long long)rows * (cols + pad);
    hipLaunchKernelGGL(normalize_kernel, dim3((unsigned)std::min<long long>((n + 1023) / 1024, 1024)), dim3(256), 0, (hipStream_t)stream, a);
    ODMKV_CHECK_LAUNCH("normalize_kernel");
    return 0;
}
