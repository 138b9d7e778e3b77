// Shared host/device helpers for libodmkv (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <hip/hip_bf16.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "../../include/odmkv.h"

#define HD ODMKV_HEAD_DIM       // 128
#define TILE ODMKV_TILE         // 64
#define WAVE 64

// ---- error slot -------------------------------------------------------------------------------
void odmkv_set_error(const char* fmt, ...);

#define ODMKV_CHECK_ARG(cond, ...)                 \
    do {                                           \
        if (!(cond)) {                             \
            odmkv_set_error(__VA_ARGS__);          \
            return ODMKV_EINVAL;                   \
        }                                          \
    } while (0)

#define ODMKV_CHECK_HIP(expr)                                                        \
    do {                                                                             \
        hipError_t e_ = (expr);                                                      \
        if (e_ != hipSuccess) {                                                      \
            odmkv_set_error("%s failed: %s", #expr, hipGetErrorString(e_));          \
            return ODMKV_EHIP;                                                       \
        }                                                                            \
    } while (0)

#define ODMKV_CHECK_LAUNCH(name)                                                     \
    do {                                                                             \
        hipError_t e_ = hipGetLastError();                                           \
        if (e_ != hipSuccess) {                                                      \
            odmkv_set_error("launch of %s failed: %s", name, hipGetErrorString(e_)); \
            return ODMKV_EHIP;                                                       \
        }                                                                            \
    } while (0)

// More than 64 KB of LDS for a kernel.  The attribute belongs to the function on the current device, so it is set before every
// launch: layers of one model may live on several devices.
#define ODMKV_ALLOW_LDS(kernel, bytes) \
    ODMKV_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)(bytes)))

static inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }
// pack.hip: byte offset, inside the pack workspace, of the list of tiles the fp16 quantiser hands to the exact one
size_t pack_redo_offset(int nseg, int T);

// level index of a bit width: 0 -> evicted, 2,3,4,8 -> 1..4, 16 -> 5; anything else -> -1
__host__ __device__ static inline int level_slot(int bits) {
    switch (bits) {
        case 0: return 0;
        case 2: return 1;
        case 3: return 2;
        case 4: return 3;
        case 8: return 4;
        case 16: return 5;
        default: return -1;
    }
}
__host__ __device__ static inline int width_of(int li) { return li == 0 ? 2 : li == 1 ? 3 : li == 2 ? 4 : 8; }
// offset of width li's table inside the concatenated codebook array (4 + 8 + 16 + 256 floats)
__host__ __device__ static inline int codebook_offset(int li) { return li == 0 ? 0 : li == 1 ? 4 : li == 2 ? 12 : 28; }
#define CODEBOOK_FLOATS 284

// ---- element loads ----------------------------------------------------------------------------
template <int DT> struct Elem;
template <> struct Elem<ODMKV_F16> {
    typedef uint16_t raw;
    __device__ static inline float to_f32(uint16_t v) { return __half2float(__ushort_as_half(v)); }
    __device__ static inline uint16_t from_f32(float f) { return __half_as_ushort(__float2half_rn(f)); }
};
template <> struct Elem<ODMKV_BF16> {
    typedef uint16_t raw;
    __device__ static inline float to_f32(uint16_t v) { return __uint_as_float(((uint32_t)v) << 16); }
    __device__ static inline uint16_t from_f32(float f) {
        return __builtin_bit_cast(uint16_t, (__bf16)f);      // nearest even; one instruction on gfx950 (seven in integer arithmetic)
    }
};
template <> struct Elem<ODMKV_F32> {
    typedef float raw;
    __device__ static inline float to_f32(float v) { return v; }
    __device__ static inline float from_f32(float f) { return f; }
};

// of the current device, and what they all have if it does not say
static inline int compute_units() {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) return v;
    return 256;
}

// Wave-wide reductions (64 lanes, all of them active; every lane ends with the result) by DPP moves and lane swaps: a shuffle is a read of LDS, six of them
// one behind the other.
template <int CTRL>
__device__ static inline float wave_dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <typename F>
__device__ static inline float wave_fold(float v, F f) {
    v = f(v, wave_dpp<0xB1>(v));                          // lane ^ 1
    v = f(v, wave_dpp<0x4E>(v));                          // lane ^ 2
    v = f(v, wave_dpp<0x141>(v));                         // the other four of eight
    v = f(v, wave_dpp<0x140>(v));                         // the other eight of sixteen
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ static inline float wave_sum(float v) { return wave_fold(v, [](float x, float y) { return x + y; }); }
__device__ static inline float wave_max(float v) { return wave_fold(v, [](float x, float y) { return fmaxf(x, y); }); }
