// Shared device/host helpers for the gfx950 kernels of libcacti_gpu_hip_ffi.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/cacti_gpu_hip_ffi.h"

#define CACTI_API extern "C" __attribute__((visibility("default")))

namespace cacti {

// ---- status plumbing -------------------------------------------------------
void set_error(const char *fmt, ...);
int hip_status(hipError_t e, const char *what);

#define CACTI_HIP(expr)                                        \
    do {                                                       \
        hipError_t e_ = (expr);                                \
        if (e_ != hipSuccess) return ::cacti::hip_status(e_, #expr); \
    } while (0)

#define CACTI_REQUIRE(cond, code, ...)          \
    do {                                        \
        if (!(cond)) {                          \
            ::cacti::set_error(__VA_ARGS__);    \
            return (code);                      \
        }                                       \
    } while (0)

// State a launcher establishes once per device and keeps (a kernel's dynamic-LDS attribute, the device
// address of a file-scope array) belongs to the device's loaded modules.  cacti_hip_primary_ctx_reset
// unloads them, so it advances an epoch, and every such cache is tagged with (device, epoch) and set up
// again when either differs.
unsigned module_epoch();
void module_epoch_advance();
// device contexts (cacti_ctx) alive on a device: a primary-context reset under one would free its pool,
// streams and events behind its back, so the reset entry point refuses while any exists
int live_contexts(int dev);
void live_contexts_add(int dev, int n);
// compute units of the current device (256 where there is none)
int device_cus();
struct DeviceOnce {
    int dev = -1;
    unsigned epoch = 0;
    bool fresh() const
    {
        int d = -2;
        return hipGetDevice(&d) == hipSuccess && d == dev && epoch == module_epoch();
    }
    void mark()
    {
        if (hipGetDevice(&dev) != hipSuccess) dev = -1;
        epoch = module_epoch();
    }
};

inline int launch_status(const char *what) { return hip_status(hipGetLastError(), what); }

inline bool aligned(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

// ---- f16 <-> f32 with IEEE round-to-nearest-even ----------------------------
typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float h2f(half_t h) { return (float)h; }
__device__ __forceinline__ half_t f2h(float f) { return (half_t)f; }   // v_cvt_f16_f32, RNE
// round an fp32 value to the nearest f16 and come back: one reference thunk boundary
__device__ __forceinline__ float rnd16(float f) { return (float)(half_t)f; }

// 16-byte vector of 8 halves moved as one global/LDS transaction
struct __attribute__((aligned(16))) h8 {
    half_t v[8];
};
__device__ __forceinline__ h8 ld8(const half_t *p) { return *reinterpret_cast<const h8 *>(p); }
__device__ __forceinline__ void st8(half_t *p, const h8 &x) { *reinterpret_cast<h8 *>(p) = x; }

// ---- 64-lane wavefront reductions ------------------------------------------
// Lanes exchange without LDS: through DPP within a row of 16 (quad_perm, row_half_mirror, row_mirror), across the rows and the
// halves by v_permlane16_swap / v_permlane32_swap of a register with itself, which give both sides in every lane (an exchange
// through LDS is a hundred cycles and more, one behind another; an fp64 sum was six of two words each); every lane ends with the
// full result.  32 tokens of 3 layers of 3200 7083 -> 6968 us, a prompt of 1531 and 16 tokens of 4 layers of 2048 3916 -> 3822,
// 32 tokens of 2 layers of 256 1.8 ms on either side, against ds_swizzle and ds_bpermute for the last two steps.  T: 4 bytes
template <int CTRL, class T>
__device__ __forceinline__ T dpp(T v)
{
    return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) { return dpp<CTRL>(v); }
typedef unsigned both_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ both_t both16(unsigned v) { return __builtin_amdgcn_permlane16_swap(v, v, false, false); }
__device__ __forceinline__ both_t both32(unsigned v) { return __builtin_amdgcn_permlane32_swap(v, v, false, false); }
// op of a lane's value and that of lane ^ 16, ^ 32
template <class T, class Op>
__device__ __forceinline__ T with16(T v, Op op)
{
    const both_t b = both16(__builtin_bit_cast(unsigned, v));
    const unsigned x = b[0], y = b[1];          // (a bit cast of a vector's element takes its first)
    return op(__builtin_bit_cast(T, x), __builtin_bit_cast(T, y));
}
template <class T, class Op>
__device__ __forceinline__ T with32(T v, Op op)
{
    const both_t b = both32(__builtin_bit_cast(unsigned, v));
    const unsigned x = b[0], y = b[1];          // (a bit cast of a vector's element takes its first)
    return op(__builtin_bit_cast(T, x), __builtin_bit_cast(T, y));
}

struct OpSum {
    __device__ __forceinline__ float operator()(float a, float b) const { return a + b; }
};
struct OpMax {
    __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); }
};

template <class T, class Op>
__device__ __forceinline__ T wave_reduce(T v, Op op)
{
    v = op(v, dpp<0xB1>(v));    // quad_perm [1,0,3,2]  : lane ^ 1
    v = op(v, dpp<0x4E>(v));    // quad_perm [2,3,0,1]  : lane ^ 2
    v = op(v, dpp<0x141>(v));   // row_half_mirror      : other quad of the 8
    v = op(v, dpp<0x140>(v));   // row_mirror           : other half of the 16
    return with32(with16(v, op), op);
}
__device__ __forceinline__ float wave_sum(float v) { return wave_reduce(v, OpSum()); }
__device__ __forceinline__ float wave_max(float v) { return wave_reduce(v, OpMax()); }

// fp64 sum over the 64 lanes, in the same steps; every lane ends with the result
__device__ __forceinline__ double words_f64(unsigned lo, unsigned hi) { return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo); }
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v)
{
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    return words_f64(__builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xf, 0xf, false),
                     __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ double wave_sum_f64(double v)
{
    v += dpp_f64<0xB1>(v);
    v += dpp_f64<0x4E>(v);
    v += dpp_f64<0x141>(v);
    v += dpp_f64<0x140>(v);
    uint64_t u = __builtin_bit_cast(uint64_t, v);
    both_t lo = both16((unsigned)u), hi = both16((unsigned)(u >> 32));
    u = __builtin_bit_cast(uint64_t, words_f64(lo[0], hi[0]) + words_f64(lo[1], hi[1]));
    lo = both32((unsigned)u);
    hi = both32((unsigned)(u >> 32));
    return words_f64(lo[0], hi[0]) + words_f64(lo[1], hi[1]);
}

// Block reduction through LDS: `red` holds one float per wave (<= 16 waves).
template <class Op>
__device__ __forceinline__ float block_reduce(float v, Op op, float ident, float *red)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    v = wave_reduce(v, op);
    __syncthreads();                // protect `red` against the previous use
    if (lane == 0) red[wid] = v;
    __syncthreads();
    float r = ident;
    for (int i = 0; i < nw; i++) r = op(r, red[i]);
    return r;
}

}  // namespace cacti
