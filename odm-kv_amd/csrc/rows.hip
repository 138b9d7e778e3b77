// Row-wise TurboQuant-MSE quantise / dequantise without the packed store.  Same codes as the tile kernels of the packed
// store: 16-bit rows of 2, 3 and 4 bits on the matrix cores (pack.hip), everything else, and what those leave, one lane per
// row in the definition's order (here).
#include <algorithm>
#include "quant.h"

// one tile of 64 rows, a row per lane; cb: the width's centroids in LDS
template <int W, int DT>
__device__ static void quantize_rows_tile(const RowsJob& job, int64_t tile, float* cb) {
    const int lane = threadIdx.x;
    for (int i = lane; i < (1 << W); i += WAVE) cb[i] = job.cb[i];
    __syncthreads();
    const int64_t n = tile * WAVE + lane;
    const bool valid = n < job.n;
    float u[HD];
    if (valid) load_row<DT>(job.x, (size_t)row_offset(job, n), u);
    else {
#pragma unroll
        for (int j = 0; j < HD; ++j) u[j] = 0.0f;
    }
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < HD; ++j) ss = __fmaf_rn(u[j], u[j], ss);
    const float norm = sqrtf(ss);
    const float den = norm + 1e-10f;
#pragma unroll
    for (int j = 0; j < HD; ++j) u[j] = u[j] / den;
    if (valid) job.norms[n] = norm;
    const int row_bytes = job.packed ? container_bytes(W) : HD;
#pragma unroll 1
    for (int i0 = 0; i0 < HD; i0 += 8) {
        float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        const float* __restrict__ rows = job.pi + (size_t)i0 * HD;
#pragma unroll
        for (int j = 0; j < HD; ++j) {
#pragma unroll
            for (int b = 0; b < 8; ++b) acc[b] = __fmaf_rn(u[j], rows[b * HD + j], acc[b]);
        }
        uint32_t w0 = 0, w1 = 0, wp = 0;                       // a byte each, and the container's bits
        constexpr int EFF = W == 3 ? 4 : W;
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint32_t c = nearest_code<W>(acc[b], cb);
            if (b < 4) w0 |= c << (8 * b); else w1 |= c << (8 * (b - 4));
            if constexpr (W < 8) wp |= c << (EFF * b);
        }
        if (!valid) continue;
        uint8_t* dst = job.codes + (size_t)n * row_bytes;
        if (W == 8 || !job.packed) *reinterpret_cast<uint2*>(dst + i0) = make_uint2(w0, w1);
        else if constexpr (W == 2) *reinterpret_cast<uint16_t*>(dst + i0 / 4) = (uint16_t)wp;
        else *reinterpret_cast<uint32_t*>(dst + i0 / 2) = wp;
    }
}

template <int W, int DT>
__global__ __launch_bounds__(64) void quantize_rows_kernel(RowsJob job) {
    __shared__ float cb[1 << W];
    quantize_rows_tile<W, DT>(job, blockIdx.x, cb);
}

// The tiles that the matrix-core quantiser has marked (rows with infinities or many values next to a threshold; usually none: the launch's own
// time counts).  A workgroup looks 64 tiles over, a lane each, and does the marked ones.
template <int DT>
__global__ __launch_bounds__(64) void quantize_flagged_rows_kernel(RowsJob job) {
    __shared__ float cb[16];
    const int64_t tile0 = (int64_t)blockIdx.x * WAVE, at = (tile0 + threadIdx.x) * WAVE;
    unsigned long long marked = __ballot(at < job.n && __float_as_uint(job.norms[at]) == ROWS_HANDED_OVER);
    while (marked) {                                           // (wave-uniform; a wavefront is the workgroup)
        const int64_t tile = tile0 + __builtin_ctzll(marked);
        marked &= marked - 1ull;
        __syncthreads();                                       // the last tile's centroids have been read
        switch (job.bits) {
            case 2: quantize_rows_tile<2, DT>(job, tile, cb); break;
            case 3: quantize_rows_tile<3, DT>(job, tile, cb); break;
            default: quantize_rows_tile<4, DT>(job, tile, cb); break;
        }
    }
}

template <int W>
__global__ __launch_bounds__(64) void dequantize_rows_kernel(const uint8_t* __restrict__ codes,
                                                             const float* __restrict__ norms, int64_t N,
                                                             const float* __restrict__ pi, const float* __restrict__ cbg,
                                                             float* __restrict__ out, int packed) {
    __shared__ float cb[1 << W];
    const int lane = threadIdx.x;
    for (int i = lane; i < (1 << W); i += WAVE) cb[i] = cbg[i];
    __syncthreads();
    const int64_t n = (int64_t)blockIdx.x * WAVE + lane;
    if (n >= N) return;
    float y[HD];
    if (W == 8 || !packed) {
        const uint4* src = reinterpret_cast<const uint4*>(codes + (size_t)n * HD);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint4 v = src[c];
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 16; ++e) y[16 * c + e] = cb[((w[e >> 2] >> (8 * (e & 3))) & 0xffu) & ((1u << W) - 1u)];
        }
    } else if constexpr (W < 8) {
        constexpr int EFF = W == 3 ? 4 : W, PER = 32 / EFF;    // container codes of a 32-bit word
        const uint4* src = reinterpret_cast<const uint4*>(codes + (size_t)n * container_bytes(W));
#pragma unroll
        for (int c = 0; c < HD / (4 * PER); ++c) {
            const uint4 v = src[c];
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 4 * PER; ++e) y[4 * PER * c + e] = cb[(w[e / PER] >> (EFF * (e % PER))) & ((1u << W) - 1u)];
        }
    }
    const float norm = norms[n];
#pragma unroll 1
    for (int j0 = 0; j0 < HD; j0 += 8) {
        float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < HD; ++i) {
#pragma unroll
            for (int b = 0; b < 8; ++b) acc[b] = __fmaf_rn(y[i], pi[i * HD + j0 + b], acc[b]);
        }
#pragma unroll
        for (int b = 0; b < 8; ++b) acc[b] = acc[b] * norm;
        store8<ODMKV_F32>(out, (size_t)n * HD + j0, acc);
    }
}

template <int W>
static void launch_exact(const RowsJob& j, int dtype, hipStream_t st) {
    const dim3 grid((unsigned)((j.n + WAVE - 1) / WAVE)), block(64);
    if (dtype == ODMKV_F16) hipLaunchKernelGGL((quantize_rows_kernel<W, ODMKV_F16>), grid, block, 0, st, j);
    else if (dtype == ODMKV_BF16) hipLaunchKernelGGL((quantize_rows_kernel<W, ODMKV_BF16>), grid, block, 0, st, j);
    else hipLaunchKernelGGL((quantize_rows_kernel<W, ODMKV_F32>), grid, block, 0, st, j);
}

static int launch_quantize_rows_exact(const RowsJob& j, int dtype, hipStream_t st) {
    switch (j.bits) {
        case 2: launch_exact<2>(j, dtype, st); break;
        case 3: launch_exact<3>(j, dtype, st); break;
        case 4: launch_exact<4>(j, dtype, st); break;
        default: launch_exact<8>(j, dtype, st); break;
    }
    ODMKV_CHECK_LAUNCH("quantize_rows_kernel");
    return 0;
}

static int check_rows(const char* who, const void* x, const float* pi, const float* cb, int dtype, int64_t N, int64_t stride_n, int bits) {
    ODMKV_CHECK_ARG(x && pi && cb, "%s: null pointer", who);
    ODMKV_CHECK_ARG(dtype == ODMKV_F16 || dtype == ODMKV_BF16 || dtype == ODMKV_F32, "%s: bad dtype %d", who, dtype);
    ODMKV_CHECK_ARG(bits == 2 || bits == 3 || bits == 4 || bits == 8, "%s: width %d not in {2,3,4,8}", who, bits);
    ODMKV_CHECK_ARG(N >= 0 && N < ((int64_t)1 << 37), "%s: bad row count", who);
    const int align = dtype == ODMKV_F32 ? 4 : 8;
    ODMKV_CHECK_ARG(stride_n % align == 0 && stride_n >= HD && ((uintptr_t)x & 15) == 0, "%s: rows must be 16-byte aligned", who);
    return 0;
}

// 16-bit rows of 2, 3 and 4 bits take the matrix cores first and the exact quantiser for what they leave
static int quantize(const RowsJob& job, int dtype, hipStream_t st) {
    if (dtype == ODMKV_F32 || job.bits == 8) return launch_quantize_rows_exact(job, dtype, st);
    if (int rc = launch_quantize_rows_f16(job, dtype, st)) return rc;
    const dim3 grid((unsigned)((job.n + WAVE * WAVE - 1) / (WAVE * WAVE))), block(WAVE);
    if (dtype == ODMKV_F16) hipLaunchKernelGGL(quantize_flagged_rows_kernel<ODMKV_F16>, grid, block, 0, st, job);
    else hipLaunchKernelGGL(quantize_flagged_rows_kernel<ODMKV_BF16>, grid, block, 0, st, job);
    ODMKV_CHECK_LAUNCH("quantize_flagged_rows_kernel");
    return 0;
}

static int quantize_rows(const char* who, const void* x, int dtype, int64_t N, int64_t stride_n, int bits, const float* pi, const float* cb,
                         uint8_t* codes, float* norms, int packed, void* stream) {
    ODMKV_CHECK_ARG(codes && norms, "%s: null pointer", who);
    if (int rc = check_rows(who, x, pi, cb, dtype, N, stride_n, bits)) return rc;
    ODMKV_CHECK_ARG(((uintptr_t)codes & 15) == 0, "%s: rows must be 16-byte aligned", who);
    if (N == 0) return 0;
    const RowsJob j = {x, 0, (long long)stride_n, (long long)N, (long long)N, bits, packed, pi, cb, codes, norms, nullptr};
    return quantize(j, dtype, (hipStream_t)stream);
}

extern "C" int odmkv_quantize_rows(const void* x, int dtype, int64_t N, int64_t stride_n, int bits,
                                   const float* pi, const float* cb, uint8_t* codes, float* norms,
                                   void* stream) {
    return quantize_rows("quantize_rows", x, dtype, N, stride_n, bits, pi, cb, codes, norms, 0, stream);
}

extern "C" int odmkv_quantize_rows_packed(const void* x, int dtype, int64_t N, int64_t stride_n, int bits,
                                          const float* pi, const float* cb, uint8_t* indices, float* norms, void* stream) {
    return quantize_rows("quantize_rows_packed", x, dtype, N, stride_n, bits, pi, cb, indices, norms, 1, stream);
}

static int dequantize_rows(const char* who, const uint8_t* codes, const float* norms, int64_t N, int bits, const float* pi,
                           const float* cb, float* out, int packed, void* stream) {
    ODMKV_CHECK_ARG(codes && norms && pi && cb && out, "%s: null pointer", who);
    ODMKV_CHECK_ARG(bits == 2 || bits == 3 || bits == 4 || bits == 8, "%s: width %d not in {2,3,4,8}", who, bits);
    ODMKV_CHECK_ARG(N >= 0 && N < ((int64_t)1 << 37), "%s: bad row count", who);
    ODMKV_CHECK_ARG(((uintptr_t)codes & 15) == 0 && ((uintptr_t)out & 15) == 0, "%s: buffers must be 16-byte aligned", who);
    if (N == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    dim3 grid((unsigned)((N + WAVE - 1) / WAVE)), block(64);
    switch (bits) {
        case 2: hipLaunchKernelGGL((dequantize_rows_kernel<2>), grid, block, 0, st, codes, norms, N, pi, cb, out, packed); break;
        case 3: hipLaunchKernelGGL((dequantize_rows_kernel<3>), grid, block, 0, st, codes, norms, N, pi, cb, out, packed); break;
        case 4: hipLaunchKernelGGL((dequantize_rows_kernel<4>), grid, block, 0, st, codes, norms, N, pi, cb, out, packed); break;
        default: hipLaunchKernelGGL((dequantize_rows_kernel<8>), grid, block, 0, st, codes, norms, N, pi, cb, out, packed); break;
    }
    ODMKV_CHECK_LAUNCH("dequantize_rows_kernel");
    return 0;
}

extern "C" int odmkv_dequantize_rows(const uint8_t* codes, const float* norms, int64_t N, int bits,
                                     const float* pi, const float* cb, float* out, void* stream) {
    return dequantize_rows("dequantize_rows", codes, norms, N, bits, pi, cb, out, 0, stream);
}

extern "C" int odmkv_dequantize_rows_packed(const uint8_t* indices, const float* norms, int64_t N, int bits,
                                            const float* pi, const float* cb, float* out, void* stream) {
    return dequantize_rows("dequantize_rows_packed", indices, norms, N, bits, pi, cb, out, 1, stream);
}

extern "C" size_t odmkv_round_trip_workspace_bytes(int64_t n) {
    return n > 0 ? 2 * (align_up((size_t)n * HD, 256) + align_up((size_t)n * sizeof(float), 256)) : 0;
}

extern "C" int odmkv_round_trip_rows(void* K, void* V, int dtype, int64_t groups, int64_t group_rows, int64_t stride_group,
                                     int64_t stride_row, int bits_k, int bits_v, const float* pi_k, const float* pi_v,
                                     const float* cb_k, const float* cb_v, void* workspace, size_t workspace_bytes, void* stream) {
    const int64_t n = groups * group_rows;
    ODMKV_CHECK_ARG(groups > 0 && group_rows > 0, "round_trip_rows: bad shape");
    ODMKV_CHECK_ARG(dtype == ODMKV_F16 || dtype == ODMKV_BF16, "round_trip_rows: 16-bit rows only");
    ODMKV_CHECK_ARG((bits_k != 8 && bits_v != 8) || (workspace && ((uintptr_t)workspace & 15) == 0 && workspace_bytes >= odmkv_round_trip_workspace_bytes(n)),
                    "round_trip_rows: workspace too small");
    RowsJob j[2];
    char* ws = (char*)workspace;                               // (8 bits: codes and norms between the two steps)
    for (int i = 0; i < 2; ++i) {
        void* x = i ? V : K;
        j[i] = {x, (long long)stride_group, (long long)stride_row, (long long)group_rows, (long long)n, i ? bits_v : bits_k, 0,
                i ? pi_v : pi_k, i ? cb_v : cb_k, nullptr, nullptr, x};
        if (int rc = check_rows("round_trip_rows", x, j[i].pi, j[i].cb, dtype, n, stride_row, j[i].bits)) return rc;
        ODMKV_CHECK_ARG(stride_group % 8 == 0, "round_trip_rows: rows must be 16-byte aligned");
        if (j[i].bits != 8) continue;
        j[i].codes = (uint8_t*)ws;
        j[i].norms = (float*)(ws + align_up((size_t)n * HD, 256));
        ws += align_up((size_t)n * HD, 256) + align_up((size_t)n * sizeof(float), 256);
    }
    // 2, 3 and 4 bits in one pass, 8 bits by the exact quantiser and the dequantiser
    RowsJob narrow[2], wide[2];
    int n_narrow = 0, n_wide = 0;
    for (int i = 0; i < 2; ++i) (j[i].bits < 8 ? narrow[n_narrow++] : wide[n_wide++]) = j[i];
    if (n_narrow)
        if (int rc = launch_round_trip_rows(narrow, n_narrow, dtype, (hipStream_t)stream)) return rc;
    if (n_wide == 0) return 0;
    for (int i = 0; i < n_wide; ++i)
        if (int rc = quantize(wide[i], dtype, (hipStream_t)stream)) return rc;
    return launch_dequantize_rows_f16(wide, n_wide, dtype, (hipStream_t)stream);
}
