// What the kernels that fetch their operand tiles straight into LDS share (gemm_mfma.hip, gemm_direct.hip): the loads, the
// layouts they leave the tiles in, and the counted wait.
#pragma once
#include "common.h"

namespace cacti {
namespace {

constexpr int BK = 64;

// what the lanes of a direct load beyond the end of K fetch
__device__ __attribute__((aligned(16))) uint4 g_zero16;

// 16 bytes from the lane's own address into LDS (lane l at m0 + 16 l)
__device__ __forceinline__ void load_lds16(uint32_t m0, const void *src)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(m0), "v"(src) : "memory");
}

// Position of 16-byte k chunk q in row r of a [row][64 k] tile: q ^ swz16(r), for fragments (v_mfma_f32_16x16x32_f16) of
// 16 rows x four 16-byte k chunks per wave instruction: one pass through LDS per read (484 GB/s per CU measured; 286 with
// the swizzle of the 32-row fragments).  Period 32 rows.
__device__ __forceinline__ int swz16(int r) { return ((r >> 2) ^ r) & 7; }

__device__ __forceinline__ const half_t *at(const half_t *base, uint32_t byte_off)
{
    return reinterpret_cast<const half_t *>(reinterpret_cast<const char *>(base) + byte_off);
}

// ---- k-contiguous operand fetched straight into LDS (global_load_lds_dwordx4: the 16 bytes
// of lane l land at LDS address M0 + 16 l, no register staging and no LDS store instruction).
// A wave fills 1 KB = 8 consecutive tile rows per instruction; the chunk swizzle of the LDS
// layout is applied on the global side: the lane at chunk position p of row r fetches k chunk
// p ^ f(r), which stays inside the row's 128-byte segment.  The loads are issued from inline
// assembly, so the compiler neither counts them nor knows that they write LDS: the kernel
// waits for them itself (vmcnt) before the barrier that publishes the tile.
template <int ROWS, int NT>
struct LoadKCD {
    static_assert(ROWS * 8 % NT == 0, "whole instructions per wave");
    static constexpr int NL = ROWS * 8 / NT;
    uint32_t off[NL];              // byte offset of the lane's chunk from (row0, k = 0)

    // (32 bits hold a lane's place in a tile: the entry points take pitches below 2^23 elements only)
    __device__ __forceinline__ void init(int64_t ld, int64_t rows_left, int64_t)
    {
        const uint32_t ld2 = (uint32_t)ld * 2;
        const int last = (int)(rows_left < ROWS ? rows_left : ROWS) - 1;
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT;
            const int r = c >> 3, q = (c & 7) ^ swz16(r);
            off[it] = (uint32_t)min(r, last) * ld2 + q * 16;
        }
    }
    // lds = byte address in LDS of the tile buffer to fill; origin = &op[row0][0]
    __device__ __forceinline__ void dma(uint32_t lds, const half_t *origin, int64_t k0) const
    {
        const half_t *base = origin + k0;
        const uint32_t wave = lds + (threadIdx.x & ~63u) * 16;
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const uint32_t m0 = __builtin_amdgcn_readfirstlane(wave + it * NT * 16);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :
                         : "s"(m0), "v"(off[it]), "s"(base)
                         : "memory");
        }
    }
    // the k tile with only `left` < BK values of k: chunks beyond them are zeros (left is a multiple of 8)
    __device__ __forceinline__ void dma_tail(uint32_t lds, const half_t *base, int left) const
    {
        const uint32_t wave = lds + (threadIdx.x & ~63u) * 16;
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT, r = c >> 3, q = (c & 7) ^ swz16(r);
            const void *src = q * 8 < left ? (const void *)at(base, off[it]) : (const void *)&g_zero16;
            load_lds16(__builtin_amdgcn_readfirstlane(wave + it * NT * 16), src);
        }
    }
    // instruction `it` of the NL alone (base = origin + k0): lets the caller place each load between MFMAs
    __device__ __forceinline__ void dma1(int it, uint32_t lds, const half_t *base) const
    {
        const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds + (threadIdx.x & ~63u) * 16 + it * NT * 16);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(m0), "v"(off[it]), "s"(base)
                     : "memory");
    }
    __device__ __forceinline__ const half_t *kbase(const half_t *origin, int64_t k0) const { return origin + k0; }
    __device__ __forceinline__ void load(uint4 *, const half_t *, int64_t) const {}
    __device__ __forceinline__ void store(const uint4 *, half_t *) const {}
    static constexpr int NREG = 1;
    static constexpr int NDMA = NL;
};

// ---- k-strided operand (memory [k][row]) fetched straight into LDS in its own layout,
// [64 k][ROWS] with the 16-byte chunks of k row k swizzled by 2 (k & 3), or 2 (k & 1) where ROWS is no multiple of 64; the MFMA fragments
// come out of it through ds_read_b64_tr_b16, which hands each lane of a 16-lane group 4
// consecutive k of one row from a 4 k x 16 rows block (the swizzle spreads the 4 k rows of such
// a block over all banks).  A wave fills 1 KB = 1024 / (2 ROWS) whole k rows per instruction.
template <int ROWS, int NT>
struct LoadKSD {
    static constexpr int CPR = ROWS / 8;           // 16-byte chunks per k row
    static constexpr int SWK = CPR % 8 == 0 ? 3 : 1;               // (the swizzle stays inside a k row)
    static_assert(BK * CPR % NT == 0 && CPR >= 8 && CPR % 4 == 0, "whole instructions per wave");
    static constexpr int NL = BK * CPR / NT;
    uint32_t off[NL];              // byte offset of the lane's chunk from (k = 0, row0)
    int64_t ld;

    __device__ __forceinline__ void init(int64_t ld_, int64_t rows_left, int64_t)
    {
        ld = ld_;
        const uint32_t ld2 = (uint32_t)ld_ * 2;
        const int last = (int)(rows_left < ROWS ? rows_left : ROWS) - 8;
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT;
            const int k = c / CPR, q = (c % CPR) ^ (2 * (k & SWK));
            off[it] = k * ld2 + min(q * 8, last) * 2;              // rows_left is a multiple of 8
        }
    }
    // lds = byte address in LDS of the tile buffer to fill; origin = &op[0][row0]
    __device__ __forceinline__ void dma(uint32_t lds, const half_t *origin, int64_t k0) const
    {
        const half_t *base = origin + k0 * ld;
        const uint32_t wave = lds + (threadIdx.x & ~63u) * 16;
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const uint32_t m0 = __builtin_amdgcn_readfirstlane(wave + it * NT * 16);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                         :
                         : "s"(m0), "v"(off[it]), "s"(base)
                         : "memory");
        }
    }
    // the k tile with only `left` < BK k rows: the rows beyond them are zeros
    __device__ __forceinline__ void dma_tail(uint32_t lds, const half_t *base, int left) const
    {
        const uint32_t wave = lds + (threadIdx.x & ~63u) * 16;
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int k = (threadIdx.x + it * NT) / CPR;
            const void *src = k < left ? (const void *)at(base, off[it]) : (const void *)&g_zero16;
            load_lds16(__builtin_amdgcn_readfirstlane(wave + it * NT * 16), src);
        }
    }
    __device__ __forceinline__ void dma1(int it, uint32_t lds, const half_t *base) const
    {
        const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds + (threadIdx.x & ~63u) * 16 + it * NT * 16);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(m0), "v"(off[it]), "s"(base)
                     : "memory");
    }
    __device__ __forceinline__ const half_t *kbase(const half_t *origin, int64_t k0) const { return origin + k0 * ld; }
    __device__ __forceinline__ void load(uint4 *, const half_t *, int64_t) const {}
    __device__ __forceinline__ void store(const uint4 *, half_t *) const {}
    static constexpr int NREG = 1;
    static constexpr int NDMA = NL;
};

typedef int int4_t __attribute__((ext_vector_type(4)));
// the same at any address of a half (global memory serves it in one instruction)
typedef int int4_any __attribute__((ext_vector_type(4), aligned(2)));

// the 8 halves of v moved down by s places (s >= 0), zeros behind them
__device__ __forceinline__ int4_t halves_down(int4_t v, int s)
{
    typedef unsigned long long u64;
    const u64 lo = (u64)(uint32_t)v.y << 32 | (uint32_t)v.x, hi = (u64)(uint32_t)v.w << 32 | (uint32_t)v.z;
    const int b = (s & 3) * 16;
    const u64 l = lo >> b | (hi << 1) << (63 - b), h = hi >> b;
    const u64 x = s >= 8 ? 0 : s >= 4 ? h : l, y = s >= 4 ? 0 : h;
    return int4_t{(int)(uint32_t)x, (int)(x >> 32), (int)(uint32_t)y, (int)(y >> 32)};
}

// ---- operands of any alignment, through registers into the same layouts: lane l of the workgroup's load `it` holds what the
// direct loads bring to LDS byte 16 (l + it NT) of the tile.  What would reach beyond a row's end is read from 8 halves
// before it and moved down (rows of at least 8 halves), so that nothing outside the operand is touched.
template <int ROWS, int NT>
struct LoadKCR {
    static constexpr int NL = ROWS * 8 / NT;
    uint32_t off[NL];
    __device__ __forceinline__ void init(int64_t ld, int64_t rows_left, int64_t)
    {
        const uint32_t ld2 = (uint32_t)ld * 2;
        const int last = (int)(rows_left < ROWS ? rows_left : ROWS) - 1;
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT, r = c >> 3;
            off[it] = (uint32_t)min(r, last) * ld2 + ((c & 7) ^ swz16(r)) * 16;
        }
    }
    __device__ __forceinline__ void load(int4_t *v, const half_t *base) const
    {
#pragma unroll
        for (int it = 0; it < NL; it++) v[it] = *reinterpret_cast<const int4_any *>(at(base, off[it]));
    }
    // the k tile with only `left` < BK values of k, which end the row
    __device__ __forceinline__ void load_tail(int4_t *v, const half_t *base, int left) const
    {
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT, q = ((c & 7) ^ swz16(c >> 3)) * 8, s = max(q + 8 - left, 0);
            v[it] = halves_down(*reinterpret_cast<const int4_any *>(at(base, off[it]) - s), s);
        }
    }
    __device__ __forceinline__ const half_t *kbase(const half_t *origin, int64_t k0) const { return origin + k0; }
};
template <int ROWS, int NT>
struct LoadKSR {
    static constexpr int CPR = ROWS / 8, SWK = CPR % 8 == 0 ? 3 : 1, NL = BK * CPR / NT;
    uint32_t off[NL];
    int64_t ld;
    int down[NL];
    bool edge;
    __device__ __forceinline__ void init(int64_t ld_, int64_t rows_left, int64_t)
    {
        ld = ld_;
        edge = rows_left < ROWS;
        const uint32_t ld2 = (uint32_t)ld_ * 2;
        const int left = (int)(rows_left < ROWS ? rows_left : ROWS);
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT, k = c / CPR, q = ((c % CPR) ^ (2 * (k & SWK))) * 8;
            down[it] = max(q + 8 - left, 0);
            off[it] = k * ld2 + (q - down[it]) * 2;               // (may lie before the tile's first column: inside the row)
        }
    }
    __device__ __forceinline__ int4_t in_place(const int4_t &v, int it) const { return edge ? halves_down(v, down[it]) : v; }
    __device__ __forceinline__ void load(int4_t *v, const half_t *base) const
    {
#pragma unroll
        for (int it = 0; it < NL; it++)
            v[it] = *reinterpret_cast<const int4_any *>(reinterpret_cast<const char *>(base) + (int32_t)off[it]);
    }
    __device__ __forceinline__ void load_tail(int4_t *v, const half_t *base, int left) const
    {
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int k = (threadIdx.x + it * NT) / CPR;
            const int64_t back = (int64_t)max(k - left + 1, 0) * ld;
            v[it] = *reinterpret_cast<const int4_any *>(reinterpret_cast<const char *>(base - back) + (int32_t)off[it]);
            if (back) v[it] = int4_t{0, 0, 0, 0};
        }
    }
    __device__ __forceinline__ const half_t *kbase(const half_t *origin, int64_t k0) const { return origin + k0 * ld; }
};

// wait until at most n vector memory loads are outstanding (s_waitcnt vmcnt only)
template <int N>
__device__ __forceinline__ void wait_vmem()
{
    static_assert(N >= 0 && N < 64, "vmcnt has 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

typedef __fp16 fp16x4_t __attribute__((__vector_size__(4 * sizeof(__fp16))));

// 4 consecutive k of this lane's row out of a [k][row] tile (ds_read_b64_tr_b16)
__device__ __forceinline__ uint2 lds_read_tr(const unsigned char *q)
{
    typedef __attribute__((address_space(3))) fp16x4_t *lds_ptr;
    const fp16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_ptr)q);
    uint2 r;
    __builtin_memcpy(&r, &v, 8);
    return r;
}

}  // namespace
}  // namespace cacti
