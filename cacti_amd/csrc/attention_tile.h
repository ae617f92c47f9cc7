// What the attention kernels share (attention.hip, attention_short.hip): the arguments, the LDS tiles and how they are filled,
// the products on them, and the arithmetic between the rounding points.
#pragma once
#include "common.h"
#include "softmax_math.h"

#include <type_traits>

namespace cacti {

struct AttnArgs {
    int S, H, Dh;
    int64_t ld;
    float alpha;
    const half_t *q, *k, *v, *dO;
    const half_t *o;                     // the forward output (adjoint only; may be null)
    half_t *out, *dq, *dk, *dv;
    float *m, *l;                        // [H][S] row maximum and sum (forward output)
    float *y, *sig;                      // [H][S] adjoint scratch: sigma, and 1 / l (exact arithmetic) or the
                                         // exponent offset m log2(e) + log2(l) (fast arithmetic) of each row
    int acc_dq, acc_dk, acc_dv;
    int split, per;                      // dK / dV in parts (SPLIT): the parts' number, and the query tiles of each
    float *part;                         // [split][2: dK, dV][H][S][Dh] sums of the parts
};

namespace {

constexpr int kDP = 128;                 // padded head dim of an LDS tile
constexpr int kRowB = kDP * 2;           // bytes per tile row
constexpr int kTileRows = 64;
constexpr int kTileB = kTileRows * kRowB;   // 16 KB
constexpr int kNT = 256;                 // threads of a wave group (4 waves): the unit that loads a tile
constexpr int kBM = 128;                 // rows of the fixed operand per wave group (32 per wave)
constexpr float kSpread = 8.f;           // least row sum of exponentials for the short form of sigma (dQ kernel)

typedef __fp16 fp16x4_t __attribute__((__vector_size__(4 * sizeof(__fp16))));
// pointers into device memory, said so: inside a function that is not inlined into the kernel the
// compiler would otherwise use flat loads, which also count as LDS operations when it waits for one
typedef const __attribute__((address_space(1))) half_t *gptr_t;
typedef const __attribute__((address_space(1))) float *gfptr_t;
__device__ __forceinline__ gptr_t gp(const half_t *q) { return (gptr_t)q; }
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
// 8 bytes from device memory
__device__ __forceinline__ uint2 gload8(gptr_t q)
{
    const u32x2_t t = *(const __attribute__((address_space(1))) u32x2_t *)q;
    return make_uint2(t.x, t.y);
}

__device__ __forceinline__ int gsw(int r) { return ((r & 3) << 1) | ((r >> 2) & 1) | ((r & 8) ^ ((r & 1) << 3)); }
__device__ __forceinline__ int toff(int r, int c) { return r * kRowB + ((c ^ gsw(r)) << 4); }

__device__ __forceinline__ uint2 lds_read_tr(const unsigned char *q)
{
    typedef __attribute__((address_space(3))) fp16x4_t *lds_ptr;
    const fp16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_ptr)q);
    uint2 r;
    __builtin_memcpy(&r, &v, 8);
    return r;
}

__device__ __forceinline__ half8_t as_h8(uint2 lo, uint2 hi)
{
    const uint4 v = make_uint4(lo.x, lo.y, hi.x, hi.y);
    half8_t f;
    __builtin_memcpy(&f, &v, 16);
    return f;
}

// The K / V (Q / dO) tiles through registers into LDS: the path for tensors whose tiles cannot be loaded
// straight into LDS (DmaTileMap further down).

// 16 bytes from device memory at an address that is only 8-byte aligned (the heads of a [S, H, 100]
// tensor start every 200 bytes): one global_load_dwordx4, which needs dword alignment only
typedef uint32_t u32x4_a8_t __attribute__((ext_vector_type(4), aligned(8)));
__device__ __forceinline__ uint4 gload16(gptr_t q)
{
    const u32x4_a8_t v = *reinterpret_cast<const __attribute__((address_space(1))) u32x4_a8_t *>(q);
    return make_uint4(v.x, v.y, v.z, v.w);
}

// Per-lane constants of the mapping between a 64 x Dh tile of a [S, H, Dh] tensor and its LDS tile, for
// the 256 lanes of one wave group: piece `it` of a lane (16 bytes, 4 per lane) is row r0 + 16 it,
// columns 8 pc .. 8 pc + 7, r0 = lane / 16, pc = lane % 16.  Its element offset from the tile's first
// row is goff0 + 16 it ld (a wave-uniform step), its byte offset in the LDS tile loff + 4096 it (16
// more rows leave the chunk swizzle g(r) as it is).  A memory instruction costs the address unit the
// same for 8 as for 16 bytes per lane, and the address unit, not the arithmetic, is what these kernels
// wait for: 4 loads per tile and lane instead of 8.  Lanes whose columns lie beyond the head load a
// duplicate and store nothing: the pad columns of every tile buffer are zeroed once when the kernel
// starts.  The piece that straddles the end of the head (Dh % 8 = 4: columns Dh - 4 .. Dh + 3) is
// loaded 4 columns early, so that it stays inside the head, and shifted into place.
struct FastTileMap {
    unsigned goff0, loff;
    int r0, gcol;
    int64_t ld;
    bool colok, tail, narrow;                            // narrow: a head of 4 columns, one 8-byte piece per row
    __device__ __forceinline__ FastTileMap(int64_t ld_, int Dh, int)
    {
        const int t = threadIdx.x & (kNT - 1), pc = t & 15;
        r0 = t >> 4;
        ld = ld_;
        narrow = Dh < 8;
        colok = pc * 8 < Dh;
        tail = !narrow && colok && pc * 8 + 8 > Dh;
        gcol = narrow ? 0 : tail ? Dh - 8 : min(pc * 8, Dh - 8);
        goff0 = (unsigned)(r0 * ld_ + gcol);
        loff = (unsigned)toff(r0, pc);
    }
};

__device__ __forceinline__ void zero_lds(unsigned char *smem, int bytes)
{
    for (int o = threadIdx.x * 16; o < bytes; o += blockDim.x * 16) *reinterpret_cast<uint4 *>(smem + o) = make_uint4(0, 0, 0, 0);
    __syncthreads();
}
// The same for tiles that are loaded straight into LDS: only the chunks no load writes (window chunks nch .. 15 of
// every row), without a barrier of its own -- the loads of the first tiles are already in flight when this runs
// and touch none of these chunks; the barrier that publishes those tiles publishes the zeros.
__device__ __forceinline__ void zero_pads(unsigned char *smem, int rows, int nch)
{
    const int npad = 16 - nch;
    for (int i = threadIdx.x; i < rows * npad; i += blockDim.x) {
        const int r = i / npad, c = nch + i % npad;
        *reinterpret_cast<uint4 *>(smem + toff(r, c)) = make_uint4(0, 0, 0, 0);
    }
}

// 64 rows x Dh of a [S, H, Dh] tensor -> registers -> LDS tile, by the 256 lanes of one wave group, with
// the constants above (the forward and the dK / dV kernel; the dQ kernel has no registers to spare for
// it -- it spills 56 registers with it -- and uses the 8-byte form further down).
// Whole tiles take the straight path: 4 loads at a lane-constant offset from 4 uniform row pointers, 4
// stores at a lane-constant LDS address with immediate offsets.  The last tile of a ragged sequence
// clamps its rows and zeroes the ones beyond the end.
struct FastTileLoader {
    static constexpr int NP = kTileRows * 16 / kNT;      // 16-byte pieces per lane
    uint4 v[NP];
    int rows;                                            // rows of the tile inside the tensor (uniform)
    // src = &X[row0][head column 0]; rows_left = S - row0 >= 1
    __device__ __forceinline__ void load(const FastTileMap &m, gptr_t src, int rows_left, unsigned char *)
    {
        rows = __builtin_amdgcn_readfirstlane(min(rows_left, kTileRows));
        if (m.narrow) {
#pragma unroll
            for (int it = 0; it < NP; it++) {
                const uint2 a = gload8(src + (int64_t)min(m.r0 + 16 * it, rows - 1) * m.ld);
                v[it] = make_uint4(a.x, a.y, 0u, 0u);
            }
        } else if (rows == kTileRows) {
#pragma unroll
            for (int it = 0; it < NP; it++) v[it] = gload16(src + (int64_t)(16 * it) * m.ld + m.goff0);
        } else {
#pragma unroll
            for (int it = 0; it < NP; it++) v[it] = gload16(src + (int64_t)min(m.r0 + 16 * it, rows - 1) * m.ld + m.gcol);
        }
    }
    // the straddling piece moves into place by four selects per piece and the test for a ragged tile is
    // made once (a shuffle under a lane mask per piece took five times the instructions: forward and
    // dK / dV kernel -4 us each)
    __device__ __forceinline__ void store(const FastTileMap &m, unsigned char *tile) const
    {
        if (!m.colok) return;
        if (rows == kTileRows) {
#pragma unroll
            for (int it = 0; it < NP; it++) {
                uint4 x;
                x.x = m.tail ? v[it].z : v[it].x;
                x.y = m.tail ? v[it].w : v[it].y;
                x.z = m.tail ? 0u : v[it].z;
                x.w = m.tail ? 0u : v[it].w;
                *reinterpret_cast<uint4 *>(tile + m.loff + 4096 * it) = x;
            }
        } else {
#pragma unroll
            for (int it = 0; it < NP; it++) {
                const bool in = m.r0 + 16 * it < rows;
                uint4 x;
                x.x = !in ? 0u : m.tail ? v[it].z : v[it].x;
                x.y = !in ? 0u : m.tail ? v[it].w : v[it].y;
                x.z = (!in || m.tail) ? 0u : v[it].z;
                x.w = (!in || m.tail) ? 0u : v[it].w;
                *reinterpret_cast<uint4 *>(tile + m.loff + 4096 * it) = x;
            }
        }
    }
};

// The same with 8-byte pieces (8 per lane: row r0 + 8 it, columns 4 pc .. 4 pc + 3, r0 = lane / 32,
// pc = lane % 32), for the kernel whose registers do not hold the 16-byte loader: no piece straddles the
// end of a head (Dh % 4 = 0), the chunk swizzle of rows r0 + 8 it alternates between two values.  With
// per-piece index arithmetic instead of these lane constants a tile cost 5 times the instructions
// (dQ kernel 129 -> 125 us).
struct TileMap8 {
    unsigned goff0, loff0, loff1;
    int r0, gcol;
    int64_t ld;
    bool colok;
    __device__ __forceinline__ TileMap8(int64_t ld_, int Dh, int)
    {
        const int t = threadIdx.x & (kNT - 1), pc = t & 31;
        r0 = t >> 5;
        ld = ld_;
        colok = pc * 4 < Dh;
        gcol = min(pc * 4, Dh - 4);
        goff0 = (unsigned)(r0 * ld_ + gcol);
        loff0 = (unsigned)(toff(r0, pc >> 1) + ((pc & 1) << 3));
        loff1 = (unsigned)(toff(r0 + 8, pc >> 1) + ((pc & 1) << 3)) - 8 * kRowB;
    }
};
struct TileLoader8 {
    static constexpr int NP = kTileRows * 32 / kNT;      // 8-byte pieces per lane
    uint2 v[NP];
    int rows;
    __device__ __forceinline__ void load(const TileMap8 &m, gptr_t src, int rows_left, unsigned char *)
    {
        rows = __builtin_amdgcn_readfirstlane(min(rows_left, kTileRows));
        if (rows == kTileRows) {
#pragma unroll
            for (int it = 0; it < NP; it++) v[it] = gload8(src + (int64_t)(8 * it) * m.ld + m.goff0);
        } else {
#pragma unroll
            for (int it = 0; it < NP; it++) v[it] = gload8(src + (int64_t)min(m.r0 + 8 * it, rows - 1) * m.ld + m.gcol);
        }
    }
    __device__ __forceinline__ void store(const TileMap8 &m, unsigned char *tile) const
    {
        if (!m.colok) return;
        if (rows == kTileRows) {
#pragma unroll
            for (int it = 0; it < NP; it++)
                *reinterpret_cast<uint2 *>(tile + ((it & 1) ? m.loff1 : m.loff0) + 8 * kRowB * it) = v[it];
        } else {
#pragma unroll
            for (int it = 0; it < NP; it++) {
                const bool in = m.r0 + 8 * it < rows;
                *reinterpret_cast<uint2 *>(tile + ((it & 1) ? m.loff1 : m.loff0) + 8 * kRowB * it) =
                    make_uint2(in ? v[it].x : 0u, in ? v[it].y : 0u);
            }
        }
    }
};

// Tiles straight into LDS (global_load_lds_dwordx4: the 16 bytes of lane l land at LDS address M0 + 16 l; no
// staging registers, no LDS store instructions, no selects).  The load wants 16-byte aligned addresses and the
// heads of a [S, H, Dh] tensor with Dh % 8 = 4 start on 8-byte boundaries every other head, so a head is
// addressed from the 16-byte boundary at or below its start: a *window* of ceil((Dh + shift) / 8) chunks that
// begins shift = (h Dh) % 8 elements (0 or 4) before the head.  Everything a kernel holds per head -- LDS tiles,
// the fragments of the fixed operand, accumulator columns -- is in window positions, column d of the head at
// position d + shift; the positions outside the head hold the neighbouring heads' elements in the tiles and
// zeros in the fixed operand's fragments, so they add nothing to a product over the head dimension, and output
// columns there are not stored.  (What that costs: a non-finite value in the 4 elements next to a head makes
// that head's result non-finite too, where the reference keeps it to the neighbour until the output projection
// mixes the heads.)  One instruction of a wave fills 4 tile rows; the chunk swizzle g(r) is applied on the
// global side (the lane at chunk position p of row r fetches window chunk p ^ g(r)), lanes whose chunk lies
// beyond the window stay out of the instruction, and those positions keep the zeros the kernel wrote at its
// start.  The compiler neither counts these loads nor knows that they write LDS: the kernels wait for them
// (vmcnt) before the barrier that publishes a tile.
struct DmaTileMap {
    uint32_t voff, slot;
    int r0;
    int64_t ld;
    bool act;
    __device__ __forceinline__ DmaTileMap(int64_t ld_, int Dh, int shift)
    {
        const int t = threadIdx.x & (kNT - 1), pc = t & 15;
        r0 = t >> 4;
        ld = ld_;
        const int c = pc ^ gsw(r0);                      // g(r0 + 16 it) = g(r0)
        act = c * 8 < Dh + shift;
        voff = (uint32_t)((r0 * ld_ + c * 8) * 2);
        slot = (uint32_t)(r0 * kRowB + pc * 16);
    }
};
__device__ __forceinline__ void dma16(uint32_t lds, uint32_t voff, gptr_t base)
{
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(m0), "v"(voff), "s"(base) : "memory");
}
struct DmaTileLoader {
    // src = the window's first element in the tile's first row; rows beyond the tensor are zeroed by the lanes
    // that would have fetched them
    __device__ __forceinline__ void load(const DmaTileMap &m, gptr_t src, int rows_left, unsigned char *tile) const
    {
        const int rows = __builtin_amdgcn_readfirstlane(min(rows_left, kTileRows));
        const uint32_t wave = (uint32_t)(uintptr_t)tile + ((threadIdx.x & (kNT - 1)) >> 6) * 4 * kRowB;
        if (rows == kTileRows) {
            if (m.act) {
#pragma unroll
                for (int it = 0; it < 4; it++) dma16(wave + it * 16 * kRowB, m.voff, src + (int64_t)(16 * it) * m.ld);
            }
        } else {
#pragma unroll
            for (int it = 0; it < 4; it++) {
                if (m.r0 + 16 * it < rows) {
                    if (m.act) dma16(wave + it * 16 * kRowB, m.voff, src + (int64_t)(16 * it) * m.ld);
                } else {
                    *reinterpret_cast<uint4 *>(tile + m.slot + it * 16 * kRowB) = make_uint4(0, 0, 0, 0);
                }
            }
        }
    }
    __device__ __forceinline__ void store(const DmaTileMap &, unsigned char *) const {}
};

// the barrier that publishes the tiles just loaded (and retires the ones just read)
template <bool DMA>
__device__ __forceinline__ void tile_sync()
{
    if (DMA) __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));          // vmcnt(0) alone
    __syncthreads();
}

// The fixed operand of a lane: row `row` of a [S, H, Dh] tensor as KS fragments (k step ks: the 8
// halves at positions 16 ks + 8 lh .., position = column + shift), zero outside the head and for rows beyond S
template <int KS>
__device__ __forceinline__ void load_frags(half8_t (&f)[KS], gptr_t X, int64_t ld, int row, int S, int Dh, int lh,
                                           int shift = 0)
{
    const bool rok = row < S;
    gptr_t xr = X + (int64_t)min(row, S - 1) * ld;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        const int d0 = 16 * ks + 8 * lh - shift;          // the head's column at the fragment's first position
        const bool ok0 = rok && d0 >= 0 && d0 < Dh, ok1 = rok && d0 + 4 < Dh;
        const uint2 a = gload8(xr + max(min(d0, Dh - 4), 0));
        const uint2 b = gload8(xr + min(d0 + 4, Dh - 4));
        f[ks] = as_h8(make_uint2(ok0 ? a.x : 0u, ok0 ? a.y : 0u), make_uint2(ok1 ? b.x : 0u, ok1 ? b.y : 0u));
    }
}

// The same fragments out of an LDS tile that holds the operand's rows in window positions (a tile loaded
// straight into LDS; row = the lane's row inside the tile): what lies outside the head there is the
// neighbouring heads' data, cleared here.  Rows beyond S are zero in a tile of DmaTileLoader's; in a block of attention_short.hip
// they are the last row once more, and nothing of theirs is written.
template <int KS>
__device__ __forceinline__ void frags_from_tile(half8_t (&f)[KS], const unsigned char *tile, int row, int Dh, int lh,
                                                int shift)
{
    const unsigned char *rp = tile + row * kRowB;
    const int g = gsw(row);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
        const uint4 v = *reinterpret_cast<const uint4 *>(rp + (((2 * ks + lh) ^ g) << 4));
        const int d0 = 16 * ks + 8 * lh - shift;
        const bool ok0 = d0 >= 0 && d0 < Dh, ok1 = d0 + 4 < Dh;
        f[ks] = as_h8(make_uint2(ok0 ? v.x : 0u, ok0 ? v.y : 0u), make_uint2(ok1 ? v.z : 0u, ok1 ? v.w : 0u));
    }
}

// acc = sum over d of X[row_base + .][d] Y[.][d]: X from the LDS tile (16-byte reads), Y = fixed fragments.
// PRIO: the wave runs its chain of dependent MFMAs at raised priority, so that the other wave of the SIMD
// fills the gaps of the chain with its arithmetic instead of delaying it (forward and dQ kernel -2 %; the
// dK / dV kernel has a SIMD to itself and only pays for the two extra instructions)
template <int KS, bool PRIO = true>
__device__ __forceinline__ float16_t prod_direct(const unsigned char *tile, int row_base, const half8_t (&yf)[KS],
                                                 int l32, int lh)
{
    float16_t acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
    const int row = row_base + l32;
    const unsigned char *rp = tile + row * kRowB;
    const int g = gsw(row);
    half8_t x[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) x[ks] = *reinterpret_cast<const half8_t *>(rp + (((2 * ks + lh) ^ g) << 4));
    if (PRIO) __builtin_amdgcn_s_setprio(2);
#pragma unroll
    for (int ks = 0; ks < KS; ks++) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[ks], yf[ks], acc, 0, 0, 0);
    if (PRIO) __builtin_amdgcn_s_setprio(0);
    // all fragment reads in flight before the first product (the scheduler would otherwise pair each
    // read with its use and expose the LDS latency once per k step)
    __builtin_amdgcn_sched_group_barrier(0x100, KS, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, KS, 0);
    return acc;
}

// The same product with independent vector arithmetic issued between its MFMAs (the softmax arithmetic of the
// score tile before this one): a chain of dependent MFMAs leaves the wave nothing to issue for 32 cycles per
// link, and the two waves of a SIMD do not fill each other's gaps reliably.  `work(integral_constant<i>)` is
// piece i of NP pieces of that arithmetic: piece 0 covers the latency of the fragment reads, the others follow
// the MFMAs in equal shares; scheduling barriers keep the order as written.
template <int KS, int NP, class F>
__device__ __forceinline__ float16_t prod_direct_with(const unsigned char *tile, int row_base, const half8_t (&yf)[KS],
                                                      int l32, int lh, F &&work)
{
    float16_t acc;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
    const int row = row_base + l32;
    const unsigned char *rp = tile + row * kRowB;
    const int g = gsw(row);
    half8_t x[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) x[ks] = *reinterpret_cast<const half8_t *>(rp + (((2 * ks + lh) ^ g) << 4));
    __builtin_amdgcn_sched_barrier(0);
    work(std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0);
    auto link = [&](auto ks_c) __attribute__((always_inline)) {
        constexpr int ks = decltype(ks_c)::value;
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[ks], yf[ks], acc, 0, 0, 0);
        constexpr int p0 = 1 + ks * (NP - 1) / KS, p1 = 1 + (ks + 1) * (NP - 1) / KS;
        if constexpr (p0 < p1) work(std::integral_constant<int, p0>{});
        if constexpr (p0 + 1 < p1) work(std::integral_constant<int, p0 + 1>{});
        static_assert(p1 - p0 <= 2, "at most two pieces per MFMA");
        __builtin_amdgcn_sched_barrier(0);
    };
    link(std::integral_constant<int, 0>{});
    link(std::integral_constant<int, 1>{});
    link(std::integral_constant<int, 2>{});
    link(std::integral_constant<int, 3>{});
    if constexpr (KS > 4) link(std::integral_constant<int, 4>{});
    if constexpr (KS > 5) link(std::integral_constant<int, 5>{});
    if constexpr (KS > 6) link(std::integral_constant<int, 6>{});
    if constexpr (KS > 7) link(std::integral_constant<int, 7>{});
    static_assert(KS >= 4 && KS <= 8, "4 to 8 k steps");
    return acc;
}

// acc[dt] += sum over the 32 tile rows k_base .. k_base + 31 of X[row][32 dt + .] Y[.][row]: X by
// transposing reads of the LDS tile, Y = the packed registers y0 (rows 0..15) and y1 (rows 16..31) in
// the row permutation described at the top
template <int DT>
__device__ __forceinline__ void prod_tr(float16_t (&acc)[DT], const unsigned char *tile, int k_base, half8_t y0,
                                        half8_t y1, int lane)
{
    const int a4 = (lane >> 2) & 3, b4 = lane & 3, n16 = (lane >> 4) & 1, lh = lane >> 5;
    const int colb = 16 * n16 + 4 * b4;                 // first of the lane's 4 columns inside a 32-wide tile
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
        const int r1 = k_base + 16 * kk + 4 * lh + a4, r2 = r1 + 8;
        const unsigned char *p1 = tile + r1 * kRowB + ((colb & 4) << 1);
        const unsigned char *p2 = tile + r2 * kRowB + ((colb & 4) << 1);
        const int g1 = gsw(r1), g2 = gsw(r2);
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
            const int c = (32 * dt + colb) >> 3;
            const half8_t x = as_h8(lds_read_tr(p1 + ((c ^ g1) << 4)), lds_read_tr(p2 + ((c ^ g2) << 4)));
            acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, kk ? y1 : y0, acc[dt], 0, 0, 0);
        }
    }
}

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// The same with independent vector arithmetic between its 2 DT MFMAs (NP pieces, `work(integral_constant<i>)`):
// every transposing read is issued first, scheduling barriers keep the order as written.
template <int DT, int NP, class F>
__device__ __forceinline__ void prod_tr_with(float16_t (&acc)[DT], const unsigned char *tile, int k_base, half8_t y0,
                                             half8_t y1, int lane, F &&work)
{
    const int a4 = (lane >> 2) & 3, b4 = lane & 3, n16 = (lane >> 4) & 1, lh = lane >> 5;
    const int colb = 16 * n16 + 4 * b4;
    half8_t x[2][DT];
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
        const int r1 = k_base + 16 * kk + 4 * lh + a4, r2 = r1 + 8;
        const unsigned char *p1 = tile + r1 * kRowB + ((colb & 4) << 1);
        const unsigned char *p2 = tile + r2 * kRowB + ((colb & 4) << 1);
        const int g1 = gsw(r1), g2 = gsw(r2);
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
            const int c = (32 * dt + colb) >> 3;
            x[kk][dt] = as_h8(lds_read_tr(p1 + ((c ^ g1) << 4)), lds_read_tr(p2 + ((c ^ g2) << 4)));
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, 2 * DT>([&](auto j_c) __attribute__((always_inline)) {
        constexpr int j = decltype(j_c)::value, kk = j / DT, dt = j % DT;
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[kk][dt], kk ? y1 : y0, acc[dt], 0, 0, 0);
        constexpr int p0 = j * NP / (2 * DT), p1 = (j + 1) * NP / (2 * DT);
        if constexpr (p0 < p1) work(std::integral_constant<int, p0>{});
        if constexpr (p0 + 1 < p1) work(std::integral_constant<int, p0 + 1>{});
        static_assert(p1 - p0 <= 2, "at most two pieces per MFMA");
        __builtin_amdgcn_sched_barrier(0);
    });
}

__device__ __forceinline__ half8_t pack8(const float *p)
{
    half8_t h;
#pragma unroll
    for (int i = 0; i < 8; i++) h[i] = f2h(p[i]);
    return h;
}

// exp(s - m) as every kernel here forms it (s <= m; differences below -100 count as -100, whose
// exponential is far below half an ulp of a sum that is at least 1)
__device__ __forceinline__ float exp_diff(float s, float m) { return exp_nonpos(fmaxf(s - m, -100.0f)); }

// e / l with the reciprocal y of l given (the arithmetic of RowDivide, softmax_math.h)
__device__ __forceinline__ float div_by(float e, float l, float y)
{
    const float q0 = e * y;
    return __builtin_fmaf(__builtin_fmaf(-q0, l, e), y, q0);
}
__device__ __forceinline__ float recip_refined(float l)
{
    const float y0 = __builtin_amdgcn_rcpf(l);
    return __builtin_fmaf(__builtin_fmaf(-l, y0, 1.0f), y0, y0);
}

// The f32 arithmetic between the rounding points.  EXACT: exponential with range reduction and a
// correctly rounded quotient, the arithmetic of the separate softmax kernels; FAST: v_exp_f32 of the
// scaled difference, with the division folded into the exponent (exp2_mix below; a few ulp of f32
// away, under half of the instructions).
constexpr float kLog2e = 0x1.715476p+0f;
template <bool FAST>
struct AttnMath {
    // exp(s - m) of two f32 values (merging row statistics; every score in the exact form)
    static __device__ __forceinline__ float ex(float s, float m)
    {
        if (FAST) return __builtin_amdgcn_exp2f((s - m) * kLog2e);
        return exp_diff(s, m);
    }
    // a probability in the exact form (the fast form goes through exp2_mix)
    static __device__ __forceinline__ float prob(float s, float m, float l, float y)
    {
        return div_by(exp_diff(s, m), l, y);
    }
};

// FAST arithmetic on scores that stay f16 between their rounding point and the exponent: one fused
// multiply-add that reads the f16 value (v_fma_mix_f32) forms s log2(e) - c, where c holds the row's
// maximum (and, for a probability, log2 of the row's sum as well), and v_exp_f32 does the rest.
typedef _Float16 half2v_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float exp2_mix(half_t s, float c)
{
    return __builtin_amdgcn_exp2f(__builtin_fmaf((float)s, kLog2e, -c));
}
// maximum of 16 f16 values (exact in f16), two per instruction
__device__ __forceinline__ float max16(const half_t (&h)[16])
{
    half2v_t mx = {h[0], h[1]};
#pragma unroll
    for (int e = 2; e < 16; e += 2) mx = __builtin_elementwise_max(mx, half2v_t{h[e], h[e + 1]});
    return (float)__builtin_fmaxf16(mx[0], mx[1]);
}
// 16 f32 -> f16 (round to nearest even), two per instruction
typedef float float2v_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void round16(half_t (&h)[16], const float16_t &a)
{
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
        const half2v_t t = __builtin_convertvector(float2v_t{a[e], a[e + 1]}, half2v_t);
        h[e] = t[0];
        h[e + 1] = t[1];
    }
}
// two f32 -> packed f16 (round to nearest even) as one v_cvt_pk_f16_f32, said so: left to itself the compiler
// may fold the multiplication in front into two v_fma_mixlo / mixhi_f16, which cost 4.4 ns each per SIMD where
// a multiplication costs 2.1 and this instruction 2.8 for the pair
__device__ __forceinline__ half2v_t cvt_pk(float a, float b)
{
    uint32_t u;
    asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(u) : "v"(a), "v"(b));
    half2v_t h;
    __builtin_memcpy(&h, &u, 4);
    return h;
}
// the exponent offset of a row's probabilities: m log2(e) + log2(l)
__device__ __forceinline__ float prob_shift(float m, float l)
{
    return __builtin_fmaf(m, kLog2e, __builtin_amdgcn_logf(l));
}

// a x as an f32 value of its own: the reference scales a product in f32 and rounds the result to f16, two
// roundings; written as f2h(a * x) the compiler is free to use one instruction that multiplies and rounds to f16
// once (v_fma_mixlo_f16), which differs from that in one element of some 20,000 by an f16 ulp -- and costs
// more than the multiplication and half a packed conversion
__device__ __forceinline__ float scaled(float a, float x)
{
    float t = a * x;
    asm volatile("" : "+v"(t));
    return t;
}

// 4 consecutive d of one output row: f16(scale a[0..3] [+ old])
__device__ __forceinline__ void store_row4(half_t *dst, float a0, float a1, float a2, float a3, float scale,
                                           int acc_old)
{
    const float a[4] = {a0, a1, a2, a3};
    half4_t o;
    if (acc_old) {
        const half4_t old = *reinterpret_cast<const half4_t *>(dst);
#pragma unroll
        for (int r = 0; r < 4; r++) o[r] = f2h(scaled(scale, a[r]) + h2f(old[r]));
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++) o[r] = f2h(scaled(scale, a[r]));
    }
    *reinterpret_cast<half4_t *>(dst) = o;
}

// An output tile of 128 rows leaves through LDS when the tiles are direct (16-byte aligned rows): stores in which
// every lane addresses its own row are served at about one lane per clock and CU like such loads (16 of them per
// lane and output: 4 k cycles per workgroup), whole row segments of 16 bytes per lane are not.  stage_rows: a
// wave's 32 rows as f16(scale acc), in window positions, in the layout of an operand tile; write_rows: the
// staged rows [0, rows) to memory by all threads, the head's columns only (dst = the window's first element in
// row 0).  The same values as store_row4 writes.
template <int DT>
__device__ __forceinline__ void stage_rows(unsigned char *stage, const float16_t (&acc)[DT], int row, int lh, float scale)
{
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            half4_t o;
#pragma unroll
            for (int r = 0; r < 4; r++) o[r] = f2h(scaled(scale, acc[dt][4 * q + r]));
            *reinterpret_cast<half4_t *>(stage + toff(row, 4 * dt + q) + 8 * lh) = o;
        }
}
template <int MOST = kBM>
__device__ __forceinline__ void write_rows(const unsigned char *stage, half_t *dst, int64_t ld, int rows, int Dh,
                                           int shift, int tid, int nthr)
{
    const int nch = (Dh + shift + 7) >> 3;
    for (int i = tid; i < MOST * 16; i += nthr) {
        const int row = i >> 4, c = i & 15;
        if (row >= rows || c >= nch) continue;
        const uint4 v = *reinterpret_cast<const uint4 *>(stage + toff(row, c));
        const int d0 = 8 * c - shift;                    // the head's column at the chunk's first position
        const bool lo = d0 >= 0 && d0 < Dh, hi = d0 + 4 < Dh;
        half_t *q = dst + (int64_t)row * ld + 8 * c;
        if (lo && hi) *reinterpret_cast<uint4 *>(q) = v;
        else if (lo) *reinterpret_cast<uint2 *>(q) = make_uint2(v.x, v.y);
        else if (hi) *reinterpret_cast<uint2 *>(q + 4) = make_uint2(v.z, v.w);
    }
}

}  // namespace

// attention_short.hip, for tensors whose tiles can be loaded straight into LDS; span: window positions of a head, at most 128.
// The launches come after the question whether they take it.  dq and dkv together are an adjoint, as is either with
// attention.hip's other half.
bool attention_short_fwd_takes(int64_t S, int64_t H, int64_t span);
bool attention_short_dq_takes(int64_t S, int64_t H, bool exact);
bool attention_short_dkv_takes(int64_t S, int64_t H, int64_t span, int per);
int attention_short_fwd(const AttnArgs &p, int64_t span, bool exact, hipStream_t st);
int attention_short_dq(const AttnArgs &p, int64_t span, bool exact, hipStream_t st);
int attention_short_dkv(const AttnArgs &p, int64_t span, bool exact, hipStream_t st);

}  // namespace cacti
