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
// workgroup's rows with eight requests in flight; the rows are split so that about two thousand workgroups share the
// matrix.  The torch form (conversion to fp32, mean) moved five times the bytes: 32k x 4096 fp16 250 us, here 60 us.
template <int DT>
__global__ __launch_bounds__(MN_THREADS) void mean_part_kernel(MeanArgs a) {
    constexpr int N = Vec16<DT>::N, U = 8;
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
        for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const uint4*>(p + u * step);
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

static int mean_chunk(int batch, int rows, int cols, int per_thread) {
    const long long blocks = ((cols + MN_THREADS * per_thread - 1) / (MN_THREADS * per_thread)) * (long long)batch;
    const long long chunks = std::max<long long>(1, 2048 / blocks);
    return (int)std::max<long long>(16, (rows + chunks - 1) / chunks);
}

extern "C" size_t odmkv_token_mean_workspace_bytes(int batch, int rows, int cols) {
    if (batch <= 0 || rows <= 0 || cols <= 0) return 0;
    const int chunk = std::min(mean_chunk(batch, rows, cols, 8), mean_chunk(batch, rows, cols, 4));
    return (size_t)batch * ((rows + chunk - 1) / chunk) * cols * sizeof(float);
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
