// The products of 16-byte aligned operands (every dense product of the step): both operands straight into LDS.
//
//   C[M,N] = alpha op(A) op(B) + beta C,   f16 in, fp32 MFMA accumulate, f16 out.
//
// Four waves per workgroup, each a quarter of the tile: 16-row fragments of op(A) against 16-column fragments of op(B),
// v_mfma_f32_16x16x32_f16, whose 16 x 16 results stay in accumulation registers (AGPRs).  Tiles go from 64 x 64 to 256 x
// 256; a wave of the largest holds 128 x 128 results in all 256 of its AGPRs and is alone on its SIMD.
//
// What bounds it.  Three things share a CU's time per k tile of 64: its matrix pipes (BM BN / 32 cycles), its vector memory
// path (64 bytes per cycle: 2 (BM + BN) cycles) and its LDS port (128 bytes per cycle: (BM + BN) cycles for the arriving
// tiles, twice that for the fragments of a 2 x 2 arrangement of waves).  With a quarter of the tile per wave a fragment
// read feeds BM / 32 or BN / 32 products; eight waves on a 256 x 256 tile read half as many bytes again.  From 192 x 192
// on the matrix pipes are the longest of the three, and with every CU at work the power limit is in front of them: 1616
// TFLOP/s is what this mix of products, reads and loads sustains on random operands with no dependences (256 CUs; 872 on
// 104, where it is the matrix pipes), 4096 x 4096 x 6400 runs at 1435 to 1460 by box, 8192 x 8192 x 8192 at 1465 to 1480.
//
// The compiler does not find this schedule by itself: left alone it spills (70 to 100 registers at 128 x 128 results per
// wave) and moves the loads together, and a wave that is alone on its SIMD stands still while the vector memory path works
// a burst of loads off (all 16 loads of a wave and k tile behind its barrier: 1.70 us per k tile of 256 x 256, spread over
// the k tile's products: 1.00).  So the products are inline assembly with their operands' register classes named, and the
// order in the source is the order in the binary: between any two products stand at most one load and one fragment read.
// The compiler counts no wait states from or to inline assembly: the build checks in its assembly that no accumulator is
// touched before its product is through, that no operand comes too late, and that nothing is spilled (asm_check.py).
//
// The k loop.  A k tile is two k steps of 32, its fragments two sets of registers: while the products of one step run, the
// fragments of the next are read.  One barrier per k tile, between its two steps: behind it every wave holds the tile's
// last fragments, so the tile's buffer is free, and the next tile, complete behind the same barrier, gives its first ones.
// The smaller operand has one buffer more than the other (256 x 256: three of A, two of B, all 160 KB), so that its loads
// can be issued before the barrier and the other's behind it, evenly over the whole tile.
//
// Sums are formed in one order whatever the tile (a tail of K first, then k ascending), so every shape in kShapes gives the
// same bits.  The kernel of small outputs (M32) adds its tail last and 16 values of k per instruction: those of the register
// path.
//
// Measured (median of 200 launches back to back, operands rotated over 300 MB; the kernels that this one replaces: eight
// waves with 32 x 32 blocks of the tile interleaved, accumulators left to the compiler, on tiles of 256 x 256, 256 x 192,
// 256 x 128 and 128 x 128, four on 128 x 64 and 64 x 64): 2048 x 32000 x 3200 NT 347 -> 316 us, 4096 x 4096 x 6400
// 164 -> 147, 2048 x 3200 x 8640 119 -> 110, 2048 x 3200 x 3200 48.4 -> 44.1 (160 x 192), 3200 x 3200 x 2048 TN 45.0 ->
// 42.3, 777 x 2048 x 2048 16.4 -> 12.1, 777 x 5504 x 2048 30.2 -> 21.2, 611 x 1024 x 2816 13.8 -> 10.7, 611 x 1024 x 1024
// 7.3 -> 5.9, 128 x 688 x 256 4.4 -> 3.7.
#include "common.h"
#include "gemm_internal.h"
#include "gemm_tile.h"

#include <stdio.h>

#include <algorithm>
#include <type_traits>
#include <utility>

using namespace cacti;

namespace {

// Tile buffers in LDS: D of each operand and one more of the smaller one, as many as RES workgroups per CU leave room for.
constexpr int buffers(int bm, int bn, int res)
{
    const int room = 160 * 1024 / res / (BK * 2), least = bm < bn ? bm : bn;
    const int d = (room - least) / (bm + bn);
    return d > 4 ? 4 : d;
}

// 8 halves of a row of C that starts at any address and has `left` of them from here on
__device__ __forceinline__ void store_odd(half_t *c, const int4_t &v, int64_t left)
{
    if (left >= 8) {
        *reinterpret_cast<int4_any *>(c) = v;
    } else {
        const half_t *h = reinterpret_cast<const half_t *>(&v);
#pragma unroll
        for (int j = 0; j < 7; j++)
            if (j < left) c[j] = h[j];
    }
}
__device__ __forceinline__ void load_odd(half_t *lds, const half_t *c, int64_t left)
{
    if (left >= 8) {
        *reinterpret_cast<int4_t *>(lds) = *reinterpret_cast<const int4_any *>(c);
    } else {
#pragma unroll
        for (int j = 0; j < 7; j++)
            if (j < left) lds[j] = c[j];
    }
}

// BM x BN x 64 per workgroup; wave (wm, wn) has the 16-row fragments f of op(A) at 32 f + 16 wm and of op(B) at 32 f + 16 wn.
// M32 (64 x 64): v_mfma_f32_32x32x16_f16 on one 32 x 32 block per wave and k in ascending order, its tail last.
// ANY: operands of any alignment, through registers (LoadKCR, LoadKSR), two tile buffers of each; three tiles ahead in
// registers, which is what a k tile of 64 x 64 (a quarter of a microsecond) needs to have its loads back in time.  509 x 1003 x
// 770 in three layouts: 32.2 -> 26 us against a copy to aligned rows in front.
// CHAIN: the sum of p.chain products (offsets za, zb; K a multiple of 64, at least 256), each rounded to f16 with what the ones
// before it came to, as launches one after another that accumulate into C round it, with the sum so far in registers and the
// next product's tiles on their way while the last one's are multiplied.  Launches apart cost a start and an end each (3.7 us
// with 64 x 64, 5.7 with 160 x 192), the sum's way through memory and the gap between them: three of 611 x 1024 x 1024 21.0 ->
// 14.2 us, of 777 x 2048 x 2048 41.0 -> 31.6, of 2048 x 3200 x 3200 132 -> 114; two of 2048 x 3200 x 8640 199 -> 195.
// PART: the sums of a range of k tiles, as fp32 (split_k).  With ANY also whole products (p.part null), those of more than three
// workgroups to a CU: with this branch the compiler stays at 128 registers, of which a CU holds four (asm_check.py sees to it), and
// takes 136 to 148 without.  1201 x 3001 x 65 8.9 us on three of those, 8.3 on four of these; 509 x 1003 x 770 in three layouts, one
// to a CU, 23.7 and 24.4.
template <bool TA, bool TB, int BM, int BN, int RES, bool M32, bool ANY, bool CHAIN, bool PART>
__device__ __forceinline__ void gemm_direct_tile(const GemmArgs &p, uint32_t wg)
{
    // the whole argument block in scalar registers before anything else: read field by field where the control
    // flow first wants it, it costs five dependent round trips to memory before the first operand load
    asm volatile("" ::"s"(p.M), "s"(p.N), "s"(p.K), "s"(p.alpha), "s"(p.beta), "s"(p.A), "s"(p.lda), "s"(p.sa), "s"(p.B),
                 "s"(p.ldb), "s"(p.sb), "s"(p.C), "s"(p.ldc), "s"(p.sc), "s"(p.ztab), "s"(p.odd), "s"(p.part));
    constexpr int NT = 256, D = ANY ? 2 : buffers(BM, BN, RES);   // D: tiles between a load and its use
    constexpr bool EARLY_A = BM <= BN;                            // the operand with the spare buffer
    constexpr int NBA = ANY ? 2 : D + EARLY_A, NBB = ANY ? 2 : D + !EARLY_A;
    static_assert(D >= 2 && BM % 32 == 0 && BN % 64 == 0 && (!M32 || (BM == 64 && BN == 64)), "tile shape");
    constexpr bool TR_A = TA, TR_B = !TB;                         // fragments by transposing reads
    constexpr int NA = BM / 32, NB = BN / 32;                     // fragments of a wave
    static_assert(!PART || (!M32 && !CHAIN), "parts of one product");
    const bool in_parts = PART && (!ANY || p.part);
    static_assert(!CHAIN || (!ANY && D <= 4), "the first D tiles are of the first product");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    half_t *As = reinterpret_cast<half_t *>(smem_raw);            // [NBA][BM * BK]
    half_t *Bs = As + NBA * BM * BK;                              // [NBB][BN * BK]

    int tm, tn, bz;
    p.walk.locate(wg, tm, tn, bz);
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    int nk = (int)((p.K + BK - 1) / BK), kt0 = 0;
    const int product = nk;                                       // CHAIN: k tiles of one
    if constexpr (CHAIN) nk *= p.chain;
    const int part = bz;
    if (in_parts) {
        // the "blocks of the batch" are the parts of K: the same operands, a range of k tiles each
        const int per = p.split_tiles;
        kt0 = part * per;
        nk = min(nk, kt0 + per);
        bz = 0;
    }
    int64_t za, zb, zc;
    if (__builtin_expect(p.ztab, 0)) {
        za = p.za[bz];
        zb = p.zb[bz];
        zc = p.zc[bz];
    } else {
        za = (int64_t)bz * p.sa;
        zb = (int64_t)bz * p.sb;
        zc = (int64_t)bz * p.sc;
    }
    const half_t *A = p.A + za;
    const half_t *B = p.B + zb;
    half_t *C = p.C + zc;
    // tile origins: &op[row0][0] for a k-contiguous operand, &op[0][row0] for a strided one
    const half_t *Ao = TA ? A + m0 : A + (uint64_t)(uint32_t)m0 * (uint32_t)p.lda;
    const half_t *Bo = TB ? B + (uint64_t)(uint32_t)n0 * (uint32_t)p.ldb : B + n0;

    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wid & 1, wn = wid >> 1;
    typedef typename std::conditional<TA, LoadKSD<BM, NT>, LoadKCD<BM, NT>>::type LAD;
    typedef typename std::conditional<TB, LoadKCD<BN, NT>, LoadKSD<BN, NT>>::type LBD;
    typedef typename std::conditional<TA, LoadKSR<BM, NT>, LoadKCR<BM, NT>>::type LAR;
    typedef typename std::conditional<TB, LoadKCR<BN, NT>, LoadKSR<BN, NT>>::type LBR;
    typename std::conditional<ANY, LAR, LAD>::type la;
    typename std::conditional<ANY, LBR, LBD>::type lb;
    constexpr int NLA = la.NL, NLB = lb.NL, NE = EARLY_A ? NLA : NLB, NL = EARLY_A ? NLB : NLA;
    // (the columns of a strided operand end on a multiple of 8: its width, or the padding behind it)
    la.init(p.lda, (TA && !ANY ? (p.M + 7) / 8 * 8 : p.M) - m0, p.K);
    lb.init(p.ldb, (TB || ANY ? p.N : (p.N + 7) / 8 * 8) - n0, p.K);
    const int ktail = CHAIN ? 0 : (int)(p.K % BK);
    auto lds_addr = [](const half_t *q) __attribute__((always_inline)) { return (uint32_t)(uintptr_t)q; };
    // ANY: G sets of registers, one tile of both operands each; tile t in set (t - kt0) % G
    constexpr int G = 3;
    int4_t ra[ANY ? G : 1][ANY ? NLA : 1], rb[ANY ? G : 1][ANY ? NLB : 1];
    if constexpr (ANY) {
        const bool tail = ktail && kt0 == 0;
        if (ktail) {
            if (tail) {
                la.load_tail(ra[0], la.kbase(Ao, p.K - ktail), ktail);
                lb.load_tail(rb[0], lb.kbase(Bo, p.K - ktail), ktail);
            }
            Ao = la.kbase(Ao, -BK);
            Bo = lb.kbase(Bo, -BK);
        }
        if (!tail) {
            la.load(ra[0], la.kbase(Ao, (int64_t)kt0 * BK));
            lb.load(rb[0], lb.kbase(Bo, (int64_t)kt0 * BK));
        }
#pragma unroll
        for (int u = 1; u < G; u++) {
            // (a tile that is none loads the last one again: a load inside a branch is waited for at its end)
            const int64_t k0 = (int64_t)min(kt0 + u, nk - 1) * BK;
            if (k0 == 0 && ktail) continue;
            la.load(ra[u], la.kbase(Ao, k0));
            lb.load(rb[u], lb.kbase(Bo, k0));
        }
    } else {
        // The first D tiles.  A tail of K goes first, so that every later load is of a whole tile: step t multiplies tile
        // t - 1 and step 0 the last, incomplete one.  (M32 loads it in its turn.)
        if (!M32 && ktail) {
            if (kt0 == 0) {
                la.dma_tail(lds_addr(As), la.kbase(Ao, p.K - ktail), ktail);
                lb.dma_tail(lds_addr(Bs), lb.kbase(Bo, p.K - ktail), ktail);
            }
            Ao = la.kbase(Ao, -BK);
            Bo = lb.kbase(Bo, -BK);
        }
#pragma unroll
        for (int u = 0; u < D; u++) {
            if (M32 && ktail && u == nk - 1) {
                la.dma_tail(lds_addr(As + u * BM * BK), la.kbase(Ao, p.K - ktail), ktail);
                lb.dma_tail(lds_addr(Bs + u * BN * BK), lb.kbase(Bo, p.K - ktail), ktail);
            } else if (kt0 + u < nk && (M32 || kt0 + u > 0 || !ktail)) {
                la.dma(lds_addr(As + u * BM * BK), Ao, (int64_t)(kt0 + u) * BK);
                lb.dma(lds_addr(Bs + u * BN * BK), Bo, (int64_t)(kt0 + u) * BK);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    // lane l holds row l % 16 of a fragment pair's block and columns 4 (l / 16) .. + 3
    float4_t c[NA][NB];
    float16_t c32;                                                // M32: row l % 32, columns 8 q + 4 (l / 32) .. + 3
    if constexpr (M32) {
#pragma unroll
        for (int r = 0; r < 16; r++) c32[r] = 0.f;
    } else {
#pragma unroll
        for (int a = 0; a < NA; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) c[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
    }
    const int l16 = lane & 15, kg = lane >> 4, a4 = (lane >> 2) & 3, b4 = lane & 3;
    // byte offsets in a tile of the lane's reads.  [row][k]: one per k step (the swizzle is an exclusive or), the same for all
    // fragments up to 32 rows each; [k][row]: one per parity of the fragment, up to 64 rows each two and 32 k per k step.
    auto base_kc = [&](int w, int ks) __attribute__((always_inline)) {
        const int r = w * 16 + l16;
        return r * (BK * 2) + (((ks * 4 + kg) ^ swz16(r)) << 4);
    };
    auto base_ks = [&](int w, int odd, int pitch, int swk) __attribute__((always_inline)) {
        const int chunk = odd * 4 + w * 2 + (b4 >> 1);
        return (8 * kg + a4) * pitch + ((chunk ^ (2 * (a4 & swk))) << 4) + ((b4 & 1) << 3);
    };
    int oa[2], ob[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        oa[i] = TR_A ? base_ks(wm, i, BM * 2, BM % 64 == 0 ? 3 : 1) : base_kc(wm, i);
        ob[i] = TR_B ? base_ks(wn, i, BN * 2, 3) : base_kc(wn, i);
    }
    // M32: a fragment is 32 rows of 16 k, two of them to a k step
    const int l32 = lane & 31, lh = lane >> 5;
    auto base32 = [&](bool tr, int w) __attribute__((always_inline)) {
        if (!tr) return (w * 32 + l32) * (BK * 2);
        const int chunk = (w * 32 + 16 * ((lane >> 4) & 1)) / 8 + (b4 >> 1);
        return (8 * lh + a4) * (BM * 2) + ((chunk ^ (2 * a4)) << 4) + ((b4 & 1) << 3);
    };
    const int oa32 = base32(TR_A, wm), ob32 = base32(TR_B, wn);
    auto frag_tr = [&](const unsigned char *q, int pitch) __attribute__((always_inline)) {
        const uint2 lo = lds_read_tr(q), hi = lds_read_tr(q + 4 * pitch);
        const uint4 v = make_uint4(lo.x, lo.y, hi.x, hi.y);
        half8_t f;
        __builtin_memcpy(&f, &v, 16);
        return f;
    };
    auto read_a = [&](int tile, int ks, int a) __attribute__((always_inline)) {
        if (TR_A) return frag_tr(smem_raw + tile + oa[a & 1] + ks * 32 * (BM * 2) + (a >> 1) * 128, BM * 2);
        return *reinterpret_cast<const half8_t *>(smem_raw + tile + oa[ks] + a * (32 * BK * 2));
    };
    auto read_b = [&](int tile, int ks, int b) __attribute__((always_inline)) {
        if (TR_B) return frag_tr(smem_raw + tile + ob[b & 1] + ks * 32 * (BN * 2) + (b >> 1) * 128, BN * 2);
        return *reinterpret_cast<const half8_t *>(smem_raw + tile + ob[ks] + b * (32 * BK * 2));
    };

    auto read32 = [&](bool tr, int tile, int ks, int i, int base, int w) __attribute__((always_inline)) {
        if (tr) return frag_tr(smem_raw + tile + base + (ks * 32 + i * 16) * (BM * 2), BM * 2);
        return *reinterpret_cast<const half8_t *>(smem_raw + tile + base + (((ks * 4 + i * 2 + lh) ^ swz16(w * 32 + l32)) << 4));
    };

    half8_t fa[2][NA], fb[2][NB];
    // products, reads of a step; products the reads are spread over
    constexpr int NM = M32 ? 2 : NA * NB, NU = NA + NB, RS = M32 ? NM : NM * 3 / 4;
    // read u of the NU of a k step, in the order its products want them
    auto read_u = [&](int u, int ta, int tb, int ks) __attribute__((always_inline)) {
        if constexpr (M32) {
            if (u & 1) fb[ks][u >> 1] = read32(TR_B, tb, ks, u >> 1, ob32, wn);
            else fa[ks][u >> 1] = read32(TR_A, ta, ks, u >> 1, oa32, wm);
        } else {
            if (u == 0) fa[ks][0] = read_a(ta, ks, 0);
            else if (u <= NB) fb[ks][u - 1] = read_b(tb, ks, u - 1);
            else fa[ks][u - NB] = read_a(ta, ks, u - NB);
        }
    };
    auto mfma = [&](int ks, int m) __attribute__((always_inline)) {
        if constexpr (M32)
            asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(c32) : "v"(fb[ks][m]), "v"(fa[ks][m]));
        else
            asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c[m / NB][m % NB]) : "v"(fb[ks][m % NB]), "v"(fa[ks][m / NB]));
    };
    // The products of k step KS, between them the reads of the next step (of tile ta, tb) and N loads of one operand from
    // `src` to `lds`.  (M0 is set in front of the product and read behind it: the wait state that the load wants.)
    auto step = [&](auto ks_c, auto n_c, auto a_c, int ta, int tb, const half_t *src, uint32_t lds)
                    __attribute__((always_inline)) {
        constexpr int KS = decltype(ks_c)::value, N = decltype(n_c)::value;
        constexpr bool IS_A = decltype(a_c)::value;
#pragma unroll
        for (int m = 0; m < NM; m++) {
            const int d = N > 0 && (m + 1) * N / NM > m * N / NM ? m * N / NM : -1;
            if (d >= 0) {
                const uint32_t off = IS_A ? la.off[d > 0 && d < NLA ? d : 0] : lb.off[d > 0 && d < NLB ? d : 0];
                if constexpr (M32)
                    asm volatile("s_add_u32 m0, %5, %6\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %3, %4"
                                 : "+a"(c32)
                                 : "v"(fb[KS][m]), "v"(fa[KS][m]), "v"(off), "s"(src), "s"(lds), "i"(d * NT * 16)
                                 : "memory", "scc");
                else
                    asm volatile("s_add_u32 m0, %5, %6\n\tv_mfma_f32_16x16x32_f16 %0, %1, %2, %0\n\tglobal_load_lds_dwordx4 %3, %4"
                                 : "+a"(c[m / NB][m % NB])
                                 : "v"(fb[KS][m % NB]), "v"(fa[KS][m / NB]), "v"(off), "s"(src), "s"(lds), "i"(d * NT * 16)
                                 : "memory", "scc");
            } else {
                mfma(KS, m);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = m * NU / RS; u < (m + 1) * NU / RS && u < NU; u++) read_u(u, ta, tb, KS ^ 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    typedef std::integral_constant<int, 0> K0;
    typedef std::integral_constant<int, 1> K1;

    // alpha times the sum, rounded to fp32 (the empty asm keeps the compiler from fusing the product with the conversion
    // behind it in some of the kernels and not in others)
    auto scaled = [&](int a, int b, int r) __attribute__((always_inline)) {
        float v;
        if constexpr (M32) v = p.alpha * c32[b * 4 + r];
        else v = p.alpha * c[a][b][r];
        asm("" : "+v"(v));
        return v;
    };
    // M32: four groups q of a lane's columns in place of the fragments
    constexpr int EA = M32 ? 1 : NA, EB = M32 ? 4 : NB;
    // the accumulators are read by vector instructions from here on, which do not wait for a product by themselves
    auto sums_done = [&]() __attribute__((always_inline)) {
        asm volatile("s_nop 15\n\ts_nop 15");
        if constexpr (M32) {
            asm volatile("" : "+a"(c32));
        } else {
#pragma unroll
            for (int a = 0; a < NA; a++)
#pragma unroll
                for (int b = 0; b < NB; b++) asm volatile("" : "+a"(c[a][b]));
        }
    };
    // CHAIN: what the products before came to (at first -0, to which anything adds as itself)
    half4_t sum[CHAIN ? EA : 1][CHAIN ? EB : 1];
    if constexpr (CHAIN)
#pragma unroll
        for (int a = 0; a < EA; a++)
#pragma unroll
            for (int b = 0; b < EB; b++)
#pragma unroll
                for (int r = 0; r < 4; r++) sum[a][b][r] = (half_t)-0.0f;
    auto fold = [&]() __attribute__((always_inline)) {
        sums_done();
#pragma unroll
        for (int a = 0; a < EA; a++)
#pragma unroll
            for (int b = 0; b < EB; b++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    sum[CHAIN ? a : 0][CHAIN ? b : 0][r] = f2h(scaled(a, b, r) + h2f(sum[CHAIN ? a : 0][CHAIN ? b : 0][r]));
        // zeroed where they are, by a product of zeros: as values that the compiler assigns they get registers of their own, which
        // the loop's are copied into on its other path.  (Behind it the compiler may still move one.)
        half8_t zero;
#pragma unroll
        for (int i = 0; i < 8; i++) zero[i] = (half_t)0.0f;
        asm volatile("s_nop 4" : "+v"(zero));
        if constexpr (M32) {
            asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %1, 0" : "+a"(c32) : "v"(zero));
        } else {
#pragma unroll
            for (int a = 0; a < NA; a++)
#pragma unroll
                for (int b = 0; b < NB; b++) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %1, 0" : "+a"(c[a][b]) : "v"(zero));
        }
        sums_done();
    };

    constexpr int TA_BYTES = BM * BK * 2, TB_BYTES = BN * BK * 2, B0 = NBA * TA_BYTES;
    int ta = 0, tb = B0;                                          // byte offsets in LDS of tile t
    auto next_a = [&](int q) __attribute__((always_inline)) { return q == (NBA - 1) * TA_BYTES ? 0 : q + TA_BYTES; };
    auto next_b = [&](int q) __attribute__((always_inline)) { return q == B0 + (NBB - 1) * TB_BYTES ? B0 : q + TB_BYTES; };
    if constexpr (ANY) {
        auto store = [&](int set, int ta, int tb) __attribute__((always_inline)) {
#pragma unroll
            for (int it = 0; it < NLA; it++) {
                int4_t v = ra[set][it];
                if constexpr (TA) v = la.in_place(v, it);
                *reinterpret_cast<int4_t *>(smem_raw + ta + (threadIdx.x + it * NT) * 16) = v;
            }
#pragma unroll
            for (int it = 0; it < NLB; it++) {
                int4_t v = rb[set][it];
                if constexpr (!TB) v = lb.in_place(v, it);
                *reinterpret_cast<int4_t *>(smem_raw + tb + (threadIdx.x + it * NT) * 16) = v;
            }
        };
        // tile t + 1 moves from its set to the buffers of tile t - 1, whose fragments every wave has held since the last
        // barrier, and tile t + 1 + G is requested into the set
        auto body = [&](int set, int t, bool more) __attribute__((always_inline)) {
            const int na = next_a(ta), nb = next_b(tb);
            store(set, na, nb);
            if (more) {
                const int64_t k0 = (int64_t)(t + 1 + G) * BK;
                la.load(ra[set], la.kbase(Ao, k0));
                lb.load(rb[set], lb.kbase(Bo, k0));
            }
            __builtin_amdgcn_sched_barrier(0);
            step(K0{}, std::integral_constant<int, 0>{}, std::false_type{}, ta, tb, nullptr, 0);
            __syncthreads();
            step(K1{}, std::integral_constant<int, 0>{}, std::false_type{}, na, nb, nullptr, 0);
            ta = na;
            tb = nb;
        };
        store(0, ta, tb);
        if (kt0 + G < nk) {
            la.load(ra[0], la.kbase(Ao, (int64_t)(kt0 + G) * BK));
            lb.load(rb[0], lb.kbase(Bo, (int64_t)(kt0 + G) * BK));
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NU; u++) read_u(u, ta, tb, 0);
        int t = kt0;
        for (; t + 2 * G < nk; t += G)
#pragma unroll
            for (int u = 0; u < G; u++) body((u + 1) % G, t + u, true);
        for (; t + 1 < nk; t += G)
#pragma unroll
            for (int u = 0; u < G; u++)
                if (t + u + 1 < nk) body((u + 1) % G, t + u, t + u + 1 + G < nk);
        step(K0{}, std::integral_constant<int, 0>{}, std::false_type{}, ta, tb, nullptr, 0);
#pragma unroll
        for (int m = 0; m < NM; m++) mfma(1, m);
    } else {
    if (kt0 + D <= nk) wait_vmem<(D - 1) * (NLA + NLB)>();        // the first tile; the others stay in flight
    else wait_vmem<0>();
    __syncthreads();
#pragma unroll
    for (int u = 0; u < NU; u++) read_u(u, ta, tb, 0);
    const uint32_t wave16 = lds_addr(As) + wid * 1024;
    int t = kt0;
    const half_t *asrc = la.kbase(Ao, (int64_t)(kt0 + D) * BK), *bsrc = lb.kbase(Bo, (int64_t)(kt0 + D) * BK);
    const int64_t astep = TA ? BK * p.lda : BK, bstep = TB ? BK : BK * p.ldb;
    int te = EARLY_A ? D * TA_BYTES : B0 + D * TB_BYTES;          // buffer of tile t + D of the early operand
    // CHAIN: tiles of the present product that are still to be loaded and to be multiplied
    int to_load = product - D, to_sum = product, next = 0;
    auto next_product = [&]() __attribute__((always_inline)) {
        next++;
        to_load = product;
        if (next < p.chain) {
            asrc = Ao + p.za[next];
            bsrc = Bo + p.zb[next];
        }
    };
    if (CHAIN && to_load == 0) next_product();
    const int nk_whole = M32 && ktail ? nk - 1 : nk;
    for (; t + D < nk_whole; t++) {
        step(K0{}, std::integral_constant<int, NE>{}, std::integral_constant<bool, EARLY_A>{}, ta, tb, EARLY_A ? asrc : bsrc,
             te + wave16);
        const int na = next_a(ta), nb = next_b(tb);
        const uint32_t late = (EARLY_A ? tb : ta) + wave16;
        wait_vmem<NE + (D - 2) * (NLA + NLB)>();                  // tile t + 1 has landed
        __syncthreads();
        step(K1{}, std::integral_constant<int, NL>{}, std::integral_constant<bool, !EARLY_A>{}, na, nb, EARLY_A ? bsrc : asrc, late);
        ta = na;
        tb = nb;
        te = EARLY_A ? next_a(te) : next_b(te);
        asrc += astep;
        bsrc += bstep;
        if constexpr (CHAIN) {
            if (--to_load == 0) next_product();
            if (--to_sum == 0) {
                fold();
                to_sum = product;
            }
        }
    }
    for (; t + 1 < nk; t++) {                                     // the last tiles: nothing left to load but M32's tail
        const bool tail = M32 && ktail && t + D == nk - 1;
        if (tail) {
            if (EARLY_A) la.dma_tail(lds_addr(As) + te, la.kbase(Ao, p.K - ktail), ktail);
            else lb.dma_tail(lds_addr(As) + te, lb.kbase(Bo, p.K - ktail), ktail);
        }
        step(K0{}, std::integral_constant<int, 0>{}, std::false_type{}, ta, tb, nullptr, 0);
        const int na = next_a(ta), nb = next_b(tb);
        wait_vmem<0>();
        __syncthreads();
        if (tail) {
            if (EARLY_A) lb.dma_tail(lds_addr(As) + tb, lb.kbase(Bo, p.K - ktail), ktail);
            else la.dma_tail(lds_addr(As) + ta, la.kbase(Ao, p.K - ktail), ktail);
        }
        step(K1{}, std::integral_constant<int, 0>{}, std::false_type{}, na, nb, nullptr, 0);
        ta = na;
        tb = nb;
    }
    step(K0{}, std::integral_constant<int, 0>{}, std::false_type{}, ta, tb, nullptr, 0);
#pragma unroll
    for (int m = 0; m < NM; m++) mfma(1, m);
    }
    sums_done();

    if (in_parts) {
        // a lane's 4 consecutive columns of a row are 16 bytes of the part, four lanes a 64-byte run
        float *out = p.part + part * p.M * p.ldp;
#pragma unroll
        for (int a = 0; a < NA; a++) {
            const int64_t m = m0 + a * 32 + wm * 16 + l16;
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const int64_t n = n0 + b * 32 + wn * 16 + kg * 4;
                if (m < p.M && n < p.N) *reinterpret_cast<float4_t *>(out + m * p.ldp + n) = c[a][b];
            }
        }
        return;
    }
    __syncthreads();                                              // every wave is done with the operand buffers

    // Epilogue through LDS: the f16 tile as Cs[row][BN], 16-byte chunks swizzled by the row, leaves as whole contiguous
    // rows.  With beta the old tile is fetched into it first, so alpha acc + beta C is rounded to f16 exactly once.
    half_t *Cs = reinterpret_cast<half_t *>(smem_raw);
    constexpr int CPRC = BN / 8;                                  // chunks per row
    constexpr int CSW = (CPRC & (CPRC - 1)) == 0 ? CPRC - 1 : 7;  // swizzle mask: a power of two of them, inside a row
    constexpr int NC = BM * CPRC / NT;
    static_assert(CPRC % (CSW + 1) == 0 && BM * CPRC % NT == 0, "whole rounds of chunks");
    // (as a value the compiler cannot trace back: the addresses below are otherwise computed before the k loop)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const bool inside = m0 + BM <= p.M && n0 + BN <= p.N;
    half_t *const Ct = C + m0 * p.ldc + n0;
    if (p.beta != 0.f && p.odd) {
#pragma unroll 4
        for (int i = 0; i < NC; i++) {
            const int q = tid + i * NT, row = q / CPRC, cc = q % CPRC;
            if (m0 + row < p.M) load_odd(Cs + row * BN + ((cc ^ (row & CSW)) << 3), Ct + row * p.ldc + cc * 8, p.N - n0 - cc * 8);
        }
        __syncthreads();
    } else if (p.beta != 0.f) {
#pragma unroll 4
        for (int i = 0; i < NC; i++) {
            // chunk q of Cs holds chunk (q % CPRC) ^ (row & CSW) of its row; what lies outside C is never used
            const int q = tid + i * NT, row = q / CPRC, cc = (q % CPRC) ^ (row & CSW);
            const bool in = inside || (m0 + row < p.M && n0 + cc * 8 < p.N);
            load_lds16(lds_addr(Cs) + wid * 1024 + i * NT * 16, in ? Ct + row * p.ldc + cc * 8 : Ct);
        }
        wait_vmem<0>();
        __syncthreads();
    }
    // the lane's 4 columns of fragment (a, b): the chunk number's bits are those of b, of wn and of the lane, side by side,
    // so that the row's swizzle is an exclusive or with a constant
    const int er = M32 ? wm * 32 + (tid & 31) : wm * 16 + (tid & 15), ek = M32 ? (tid & 63) >> 5 : (tid & 63) >> 4;
    unsigned char *const eo = smem_raw + er * (BN * 2) + (ek & 1) * 8;
    const int ex = (M32 ? wn << 2 : (ek >> 1) | wn << 1) ^ (er & CSW);
    auto out4 = [&](int a, int b) __attribute__((always_inline)) {
        return reinterpret_cast<half4_t *>(eo + a * 32 * (BN * 2) + ((ex ^ (M32 ? b : b << 2)) << 4));
    };
    if (p.beta != 0.f) {
#pragma unroll
        for (int a = 0; a < EA; a++)
#pragma unroll
            for (int b = 0; b < EB; b++) {
                const half4_t old = *out4(a, b);
                half4_t o;
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = f2h(scaled(a, b, r) + p.beta * h2f(old[r]));
                *out4(a, b) = o;
            }
    } else {
#pragma unroll
        for (int a = 0; a < EA; a++)
#pragma unroll
            for (int b = 0; b < EB; b++) {
                half4_t o;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if constexpr (CHAIN) o[r] = f2h(scaled(a, b, r) + h2f(sum[a][b][r]));
                    else o[r] = f2h(scaled(a, b, r));
                }
                *out4(a, b) = o;
            }
    }
    __syncthreads();
    // a round of the workgroup copies RSTEP rows of LPR chunks, NV rounds are under way together
    constexpr int LPR = NT % CPRC == 0 ? CPRC : 8, RSTEP = NT / LPR, NR = BM / RSTEP;
    constexpr int NV = NR % 8 == 0 ? 8 : NR % 6 == 0 ? 6 : NR;
    static_assert(CPRC % LPR == 0 && CSW < LPR && BM % RSTEP == 0 && NR % NV == 0, "whole rounds");
    const int r0 = tid / LPR, cc = tid % LPR;
    const unsigned char *const co = smem_raw + r0 * (BN * 2);
    const int cx = (cc ^ (r0 & CSW)) << 4;
    // INSIDE: the tile lies wholly in C, 16-byte aligned; ODD: rows at any address, N of any length
    auto copy_out = [&](auto inside_c, auto odd_c) __attribute__((always_inline)) {
        half_t *dst = Ct + r0 * p.ldc + cc * 8;
        const int64_t step = RSTEP * p.ldc;
#pragma unroll 1
        for (int g = 0; g < CPRC / LPR; g++) {
            half_t *d = dst + g * (LPR * 8);
#pragma unroll
            for (int i0 = 0; i0 < NR; i0 += NV) {
                int4_t v[NV];
#pragma unroll
                for (int i = 0; i < NV; i++)
                    v[i] = *reinterpret_cast<const int4_t *>(co + g * (LPR * 16) + (i0 + i) * RSTEP * (BN * 2) +
                                                            (cx ^ ((((i0 + i) * RSTEP) & CSW) << 4)));
#pragma unroll
                for (int i = 0; i < NV; i++) {
                    if (decltype(odd_c)::value) {
                        if (m0 + r0 + (i0 + i) * RSTEP < p.M) store_odd(d, v[i], p.N - n0 - (g * LPR + cc) * 8);
                    } else if (decltype(inside_c)::value || (m0 + r0 + (i0 + i) * RSTEP < p.M && n0 + (g * LPR + cc) * 8 < p.N)) {
                        *reinterpret_cast<int4_t *>(d) = v[i];
                    }
                    d += step;
                }
            }
        }
    };
    if (p.odd) copy_out(std::false_type{}, std::true_type{});
    else if (inside) copy_out(std::true_type{}, std::false_type{});
    else copy_out(std::false_type{}, std::false_type{});
}

template <bool TA, bool TB, int BM, int BN, int RES, bool M32, bool ANY>
__global__ void __launch_bounds__(256, RES) gemm_direct_kernel(GemmArgs p)
{
    gemm_direct_tile<TA, TB, BM, BN, RES, M32, ANY, false, false>(p, blockIdx.x);
}
template <bool TA, bool TB, int BM, int BN, int RES, bool ANY>
__global__ void __launch_bounds__(256, RES) gemm_part_kernel(GemmArgs p)
{
    gemm_direct_tile<TA, TB, BM, BN, RES, false, ANY, false, true>(p, blockIdx.x);
}
template <int BM, int BN, int RES, bool M32>
__global__ void __launch_bounds__(256, RES) gemm_chain_kernel(GemmArgs p)
{
    gemm_direct_tile<false, false, BM, BN, RES, M32, false, true, false>(p, blockIdx.x);
}
// Two products that wait for nothing of each other, in one launch: a gradient of the inputs (NN, of a chain perhaps) and those of
// the weights (TN).  The one with the longer sums has the first workgroups, so that none of them begins when the others end; the
// other's begin at a number that keeps their XCDs.
struct PairArgs {
    uint32_t second;
    int tn_first;
    GemmArgs nn, tn;
};
template <int BM, int BN, int RES, bool M32, bool CHAIN>
__global__ void __launch_bounds__(256, RES) gemm_pair_kernel(PairArgs p)
{
    // a field of each cache line of the argument block, all requested at once: the product's own are read behind a branch
    asm volatile("" ::"s"(p.second), "s"(p.tn_first), "s"(p.nn.M), "s"(p.nn.B), "s"(p.nn.walk.full), "s"(p.nn.ztab), "s"(p.nn.zc[0]),
                 "s"(p.nn.part), "s"(p.tn.M), "s"(p.tn.B), "s"(p.tn.walk.full), "s"(p.tn.ztab), "s"(p.tn.zc[0]), "s"(p.tn.part));
    const bool first = blockIdx.x < p.second;
    const uint32_t wg = first ? blockIdx.x : blockIdx.x - p.second;
    if (first == (p.tn_first != 0)) {
        if (wg < (uint32_t)p.tn.walk.wgs) gemm_direct_tile<true, false, BM, BN, RES, M32, false, false, false>(p.tn, wg);
    } else {
        if (wg < (uint32_t)p.nn.walk.wgs) gemm_direct_tile<false, false, BM, BN, RES, M32, false, CHAIN, false>(p.nn, wg);
    }
}

// C = f16(alpha sum of the parts + beta C), four columns per lane; the parts are added in order.  VEC: N and the rows
// of C allow 8-byte accesses.  MOST: parts at most, requested together.
template <bool VEC, int MOST>
__global__ void __launch_bounds__(256)
reduce_parts_kernel(int64_t M, int64_t N, int64_t ldp, int split, const float *__restrict__ part, float alpha, float beta,
                    half_t *__restrict__ C, int64_t ldc)
{
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= M * ldp) return;
    const int64_t m = i / ldp, n = i - m * ldp;
    float4_t v[MOST];
#pragma unroll
    for (int k = 0; k < MOST; k++) v[k] = *reinterpret_cast<const float4_t *>(part + min(k, split - 1) * M * ldp + i);
    float4_t s = v[0];
#pragma unroll
    for (int k = 1; k < MOST; k++)
        if (k < split) s += v[k];
    half_t *cp = C + m * ldc + n;
    half4_t o, old = {0, 0, 0, 0};
    const bool has_beta = beta != 0.f;
    if (VEC) {
        if (has_beta) old = *reinterpret_cast<const half4_t *>(cp);
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (has_beta && n + r < N) old[r] = cp[r];
    }
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = has_beta ? f2h(alpha * s[r] + beta * h2f(old[r])) : f2h(alpha * s[r]);
    if (VEC) {
        *reinterpret_cast<half4_t *>(cp) = o;
    } else {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (n + r < N) cp[r] = o[r];
    }
}

// Operands of any alignment as operands the direct kernels take: rows of `cols` halves, `ld` apart, to rows of `out_cols`
// = cols rounded up to 8 (zeros behind cols), 16-byte aligned.  One lane per 16-byte piece, both operands in one launch.
// (One load per piece at whatever address, and results that leave in the same way: 509 x 1003 x 770 in three layouts 39.8 ->
// 32.2 us, 1999 x 3001 x 2003 152 -> 126 with the tiles of this file; half by half before.)
struct RepackArgs {
    const half_t *src[2];
    half_t *dst[2];
    int64_t rows[2], cols[2], ld[2];
};
__global__ void __launch_bounds__(256) repack_kernel(RepackArgs p)
{
    const int z = blockIdx.y;
    const int64_t per_row = (p.cols[z] + 7) / 8, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (!p.dst[z] || i >= p.rows[z] * per_row) return;
    const int64_t row = i / per_row, c = (i - row * per_row) * 8;
    const half_t *src = p.src[z] + row * p.ld[z] + c;
    const int64_t left = p.cols[z] - c;
    int4_t v = {0, 0, 0, 0};
    if (left >= 8) {
        v = *reinterpret_cast<const int4_any *>(src);
    } else {
        half_t h[8];
#pragma unroll
        for (int j = 0; j < 8; j++) h[j] = j < left ? src[j] : (half_t)0.f;
        __builtin_memcpy(&v, h, 16);
    }
    *reinterpret_cast<int4_t *>(p.dst[z] + i * 8) = v;
}

template <bool TA, bool TB, int BM, int BN, int RES, bool M32 = false, bool ANY = false, bool CHAIN = false, bool PART = false>
int launch(GemmArgs p, int64_t nblk, hipStream_t st)
{
    const int tiles_m = (int)((p.M + BM - 1) / BM), tiles_n = (int)((p.N + BN - 1) / BN);
    constexpr size_t smem = (size_t)(ANY ? 2 * (BM + BN) : buffers(BM, BN, RES) * (BM + BN) + (BM < BN ? BM : BN)) * BK * sizeof(half_t);
    void (*kern)(GemmArgs);
    if constexpr (CHAIN) kern = gemm_chain_kernel<BM, BN, RES, M32>;
    else if constexpr (PART) kern = gemm_part_kernel<TA, TB, BM, BN, RES, ANY>;
    else kern = gemm_direct_kernel<TA, TB, BM, BN, RES, M32, ANY>;
    static DeviceOnce attr_set;                   // one per instantiation
    if (!attr_set.fresh()) {
        CACTI_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        attr_set.mark();
    }
    const int64_t nwg = (int64_t)tiles_m * tiles_n * nblk;
    CACTI_REQUIRE(nwg < (int64_t)1 << 31, CACTI_E_NOTIMPL, "gemm: %lld workgroups exceed the grid limit", (long long)nwg);
    p.walk.set(tiles_m, tiles_n, gemm_walk_rows(tiles_m, tiles_n, BM, BN, nblk), nblk, p.ztab);
    hipLaunchKernelGGL(kern, dim3((unsigned)nwg), dim3(256), smem, st, p);
    return launch_status("gemm_direct");
}


// The tile shapes, and what a product costs on each in microseconds: a start and end of `fixed`, then per k tile the time of
// a full set of resident workgroups (`res` per CU: `full`), for the last, partly filled set `first` + `load` x the share of
// the CUs that are busy where no CU has more than one, and `round` for every further set.  Fitted (least squares of the
// log) to 533 of 800 products measured on MI355X: M 16 .. 8640, N 64 .. 32000, K 72 .. 16000, three layouts, half of them
// with the widths and the token counts of models.  On the other 267 the tile picked by it is 0.9 % slower in the mean than
// the best of 24 shapes tried (37 % at worst: 539 x 6736 x 1664); the best of these 14 would be 0.6 % slower.  What the ten
// others would add: 256 x 128, 128 x 256, 256 x 192, 192 x 128, 224 x 128, 64 x 256, 96 x 192, 96 x 256, 128 x 64 and four
// workgroups of 64 x 64 per CU are each the best for some product, and 1 to 3 % better than one of these there.
// (profiles/gemm_tile_times_by_shape.txt has the times.)
struct Shape {
    int bm, bn, res;                              // res: workgroups per CU
    double fixed, first, load, full, round;
};
constexpr Shape kShapes[] = {
    {64, 64, 2, 3.511, 0.183, 0.038, 0.446, 1.728},
    {96, 64, 2, 3.674, 0.209, 0.076, 0.547, 1.899},
    {160, 64, 2, 3.506, 0.406, 0.211, 0.795, 2.256},
    {64, 128, 2, 3.747, 0.245, 0.155, 0.690, 2.000},
    {96, 128, 1, 4.203, 0.286, 0.200, 0.458, 2.802},
    {128, 128, 2, 3.969, 0.425, 0.237, 0.994, 2.829},
    {128, 128, 1, 4.491, 0.326, 0.263, 0.548, 3.135},
    {160, 128, 1, 4.972, 0.368, 0.302, 0.645, 3.644},
    {128, 192, 1, 5.129, 0.430, 0.346, 0.704, 4.152},
    {160, 192, 1, 5.661, 0.500, 0.370, 0.810, 4.800},
    {192, 192, 1, 5.791, 0.567, 0.467, 0.937, 5.069},
    {160, 256, 1, 6.163, 0.627, 0.558, 1.015, 5.270},
    {192, 256, 1, 6.948, 0.733, 0.519, 1.139, 5.758},
    {256, 256, 1, 8.360, 0.901, 0.592, 1.409, 7.849},
};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);
constexpr int kChainShapes = kNumShapes - 2;      // of the last two a lane has no registers for a second sum
constexpr int T64 = 0, T64_SMALL = kNumShapes;   // T64_SMALL: 64 x 64 with M32

template <int SHAPE>
int launch_pair(const PairArgs &args, int64_t nblk, hipStream_t st)
{
    constexpr bool M32 = SHAPE == T64_SMALL;
    constexpr Shape t = kShapes[M32 ? T64 : SHAPE];
    constexpr size_t smem = (size_t)(buffers(t.bm, t.bn, t.res) * (t.bm + t.bn) + (t.bm < t.bn ? t.bm : t.bn)) * BK * sizeof(half_t);
    PairArgs p = args;
    auto kern = p.nn.chain > 1 ? gemm_pair_kernel<t.bm, t.bn, t.res, M32, true> : gemm_pair_kernel<t.bm, t.bn, t.res, M32, false>;
    static DeviceOnce attr_set;
    if (!attr_set.fresh()) {
        CACTI_HIP(hipFuncSetAttribute((const void *)gemm_pair_kernel<t.bm, t.bn, t.res, M32, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        CACTI_HIP(hipFuncSetAttribute((const void *)gemm_pair_kernel<t.bm, t.bn, t.res, M32, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        attr_set.mark();
    }
    auto set = [&](GemmArgs &g, int64_t n) {
        const int tiles_m = (int)((g.M + t.bm - 1) / t.bm), tiles_n = (int)((g.N + t.bn - 1) / t.bn);
        g.walk.set(tiles_m, tiles_n, gemm_walk_rows(tiles_m, tiles_n, t.bm, t.bn, n), n, g.ztab);
        return (int64_t)tiles_m * tiles_n * n;
    };
    p.tn_first = p.tn.K > p.nn.K * p.nn.chain;
    const int64_t wgs_nn = set(p.nn, 1), wgs_tn = set(p.tn, nblk);
    const int64_t first = ((p.tn_first ? wgs_tn : wgs_nn) + 7) / 8 * 8, second = p.tn_first ? wgs_nn : wgs_tn;
    CACTI_REQUIRE(first + second < (int64_t)1 << 31, CACTI_E_NOTIMPL, "gemm: %lld workgroups exceed the grid limit", (long long)(first + second));
    p.second = (uint32_t)first;
    hipLaunchKernelGGL(kern, dim3((unsigned)(first + second)), dim3(256), smem, st, p);
    return launch_status("gemm_pair");
}

// The tiles of a pair, both products' the same.
constexpr int kPairShapes[] = {T64_SMALL, 0, 3, 5, 7};     // 64 x 64 twice, 64 x 128, 128 x 128, 160 x 128

// The tiles that parts of K are formed on.  Of 87 products that 160 x 64 or 64 x 128 are the best for, by the costs by 2 % only, these
// take 2642 us and the next best of the others 2893 (3320 x 136 x 10176 28 and 34).  128 x 128 with two workgroups to a CU is not among
// them: where the costs put it first by 2 % it takes 6 % longer than the next (122 products; 214 x 3872 x 13944 46 and 39).  The
// remaining ones would be expected to take 0.1 % less in the mean.
constexpr bool has_parts(int tile)
{
    for (int t : {0, 1, 2, 3, 4, 6, 7, 9, 12, 13})
        if (t == tile) return true;
    return false;
}

template <bool TA, bool TB, int... I>
int launch_part_shape(int shape, const GemmArgs &p, int split, hipStream_t st, std::integer_sequence<int, I...>)
{
    if (p.any) return launch<TA, TB, 64, 64, 2, false, true, false, true>(p, split, st);
    int rc = CACTI_E_STATE;
    auto one = [&](auto i_c) {
        constexpr int i = decltype(i_c)::value;
        if constexpr (has_parts(i))
            if (shape == i) rc = launch<TA, TB, kShapes[i].bm, kShapes[i].bn, kShapes[i].res, false, false, false, true>(p, split, st);
    };
    (one(std::integral_constant<int, I>{}), ...);
    return rc;
}
int launch_parts(int ta, int tb, int shape, const GemmArgs &p, int split, hipStream_t st)
{
    const auto all = std::make_integer_sequence<int, kNumShapes>();
    if (!ta && !tb) return launch_part_shape<false, false>(shape, p, split, st, all);
    if (!ta && tb) return launch_part_shape<false, true>(shape, p, split, st, all);
    if (ta && !tb) return launch_part_shape<true, false>(shape, p, split, st, all);
    return launch_part_shape<true, true>(shape, p, split, st, all);
}

template <bool TA, bool TB, int... I>
int launch_shape(int shape, const GemmArgs &p, int64_t nblk, hipStream_t st, std::integer_sequence<int, I...>)
{
    if constexpr (!TA && !TB)
        if (p.chain > 1) {
            if (shape == T64_SMALL) return launch<TA, TB, 64, 64, 2, true, false, true>(p, nblk, st);
            int rc = CACTI_E_STATE;
            (void)((shape == I && I < kChainShapes && (rc = launch<TA, TB, kShapes[I < kChainShapes ? I : 0].bm, kShapes[I < kChainShapes ? I : 0].bn,
                                                                  kShapes[I < kChainShapes ? I : 0].res, false, false, true>(p, nblk, st), true)) || ...);
            return rc;
        }
    if (shape == T64_SMALL) return launch<TA, TB, 64, 64, 2, true>(p, nblk, st);
    if (p.any && (p.M + 63) / 64 * ((p.N + 63) / 64) * nblk > 3 * (int64_t)device_cus())
        return launch<TA, TB, 64, 64, 2, false, true, false, true>(p, nblk, st);
    if (p.any) return launch<TA, TB, 64, 64, 2, false, true>(p, nblk, st);
    int rc = CACTI_E_STATE;
    (void)((shape == I && (rc = launch<TA, TB, kShapes[I].bm, kShapes[I].bn, kShapes[I].res>(p, nblk, st), true)) || ...);
    return rc;
}

int launch_tile(int ta, int tb, int shape, const GemmArgs &p, int64_t nblk, hipStream_t st)
{
    const auto all = std::make_integer_sequence<int, kNumShapes>();
    if (!ta && !tb) return launch_shape<false, false>(shape, p, nblk, st, all);
    if (!ta && tb) return launch_shape<false, true>(shape, p, nblk, st, all);
    if (ta && !tb) return launch_shape<true, false>(shape, p, nblk, st, all);
    return launch_shape<true, true>(shape, p, nblk, st, all);
}

double tile_cost(int64_t cus, int tile, int64_t M, int64_t N, int64_t nz, int64_t ktiles)
{
    const Shape &t = kShapes[tile];
    const int64_t wg = (M + t.bm - 1) / t.bm * ((N + t.bn - 1) / t.bn) * nz, set = cus * t.res;
    const int64_t sets = wg / set;
    const double rest = (double)(wg - sets * set) / (double)cus;
    const double last = rest == 0 ? 0 : rest <= 1 ? t.first + t.load * rest : t.full;
    return t.fixed + (double)ktiles * ((double)sets * t.full + last) + t.round * (double)(sets + (rest > 0) - 1);
}

constexpr int64_t kSmallOutput = 1 << 18;
constexpr double kAnyPerTile = 1.45;
constexpr int kMostParts = 8;

// What s parts of K on tile t are expected to take (negative: there are no such parts); per_tile: factor on the time per k tile.  The
// parts and their sum cost a launch of 3 to 13 us, 2 us per million fp32 values while they are few and half of that beyond.
double part_cost(int64_t cus, int t, int64_t M, int64_t N, int64_t kt, int s, double per_tile)
{
    const int64_t per = (kt + s - 1) / s;
    if (per < 4 || (kt + per - 1) / per != s) return -1.0;                // parts of some length, none empty
    const double fixed = kShapes[t].fixed, x = (double)(M * N) * s / 1e6;
    return fixed + per_tile * (tile_cost(cus, t, M, N, s, per) - fixed) + 4.0 + (x < 4.0 ? 2.0 * x : 4.0 + x);
}

// `best` in up to kMostParts parts of K of `lent` bytes at most on tile t, if that costs less, whichever tile it was on.  A gain of 4 % on the whole product
// (`whole`) is asked of tiles above 128 x 128, whose time per k tile with a part of the CUs is the least certain (1719 x 1024 x 8256
// 39.2 -> 43.4 us without).
void split_k(int64_t cus, int t, int64_t M, int64_t N, int64_t kt, double per_tile, double whole, size_t lent, GemmPlan &best)
{
    const double margin = kShapes[t].bm * kShapes[t].bn > 128 * 128 ? 1.04 : 1.0;
    for (int s = 2; s <= kMostParts && gemm_parts_bytes(M, N, s) <= lent; s++) {
        const double c = part_cost(cus, t, M, N, kt, s, per_tile);
        if (c >= 0 && c * margin < whole && c < best.us) best = {t, T64, 0, s, c};
    }
}

// How a product is cut.  One workgroup takes one tile; a launch runs in sets of resident workgroups, and a nearly empty
// last set costs as much as a full one.  Considered: every tile shape by itself; for those of one workgroup per CU also the
// columns of the full sets in one launch and the rest on other tiles in a second (2048 x 8640 x 3200: 256 tiles of 256 x
// 256 and 448 columns); and, where the caller has a workspace (of `lent` bytes at most), up to 8 parts of K for products with fewer
// tiles than CUs and a long K, whose workgroups would otherwise run 100 k tiles one after another on a fraction of the CUs
// (37 x 3200 x 8640: 25 tiles of 64 x 64), or on small tiles, whose operands come over and over again from L2.  With parts on tiles
// to 256 x 256 and not to 128 x 128 alone, us: 2048 x 3200 x 32000 405 -> 371 (2 parts of 256 x 256 against 160 x 192), of 50000
// 656 -> 544, 2048 x 2048 x 32000 279 -> 215, 1531 x 2048 x 32000 255 -> 171, 1024 x 3200 x 32000 241 -> 192, 319 x 3200 x 27944
// 113 -> 79; of 1576 products with up to 4000 rows, widths of models and K to 50000 it changes the parts of 36, 3304 -> 2865 us.
GemmPlan make_plan(int64_t cus, int64_t M, int64_t N, int64_t K, int64_t nz, size_t lent, int shapes = kNumShapes)
{
    const int64_t kt = (K + BK - 1) / BK;
    // A small output has about 64 tiles of 64 x 64 (or one row or column of them), the shape that is best for it while they
    // run on the device all at once; more of them are cut by cost like any other product.  The device is nowhere near its
    // power limit with a small output, so the instruction is free to be the one whose sums the register path has always
    // formed.  Up to kMaxPtrBatch products in a launch go by the single product alone: a group has the bits of separate
    // launches.
    const int64_t tiles64 = (M + 63) / 64 * ((N + 63) / 64);
    const bool small = M * N <= kSmallOutput && (nz <= kMaxPtrBatch || tiles64 * nz <= kShapes[T64].res * cus);
    double best_cost = tile_cost(cus, T64, M, N, nz, kt);
    GemmPlan best = {small ? T64_SMALL : T64, T64, 0, 1, 0};
    for (int t = T64 + 1; t < shapes && !small; t++) {
        const double c = tile_cost(cus, t, M, N, nz, kt);
        if (c < best_cost) {
            best_cost = c;
            best = {t, T64, 0, 1, 0};
        }
    }
    for (int t = T64 + 1; t < shapes && !small; t++) {
        if (kShapes[t].res > 1) continue;
        const int64_t bn = kShapes[t].bn, tiles_m = (M + kShapes[t].bm - 1) / kShapes[t].bm * nz, tiles_n = (N + bn - 1) / bn;
        const int64_t cols = tiles_m * tiles_n / cus * cus / tiles_m * bn;
        if (cols <= 0 || cols >= N) continue;
        const double first = tile_cost(cus, t, M, cols, nz, kt);
        for (int r = T64; r < shapes && first < best_cost; r++) {
            const double c = first + tile_cost(cus, r, M, N - cols, nz, kt);
            if (c < best_cost) {
                best_cost = c;
                best = {t, r, cols, 1, 0};
            }
        }
    }
    best.us = best_cost;
    if (lent > 0 && nz == 1)
        for (int t = T64; t < kNumShapes; t++)
            if (has_parts(t)) split_k(cus, t, M, N, kt, 1.0, best_cost, lent, best);
    return best;
}

}  // namespace

namespace cacti {

int gemm_walk_rows(int tiles_m, int tiles_n, int bm, int bn, int64_t nblk)
{
    // An XCD works on a band of tiles / 8 consecutive tiles, i.e. on g tile rows x band / g tile columns at a time, and
    // fetches g A panels and band / g B panels per k tile into its L2: the power of two with the fewest rows fetched.
    // (Run time hardly reacts, the re-reads being served by the MALL; the L2-miss traffic does: -25 % at 2048 x 3200 x
    // 8640.)
    int rows = 8;
    if (nblk != 1) return rows;
    const double band = (double)tiles_m * tiles_n / 8.0;
    double best = 0;
    for (int g = 8; g >= 2; g /= 2) {                     // ties: the larger group
        const double fetched = g * (double)bm + band / g * (double)bn;
        if (best == 0 || fetched < best) {
            best = fetched;
            rows = g;
        }
    }
    return rows;
}

void gemm_tile_dims(int tile, int64_t *bm, int64_t *bn)
{
    const Shape &s = kShapes[tile == T64_SMALL ? T64 : tile];
    *bm = s.bm;
    *bn = s.bn;
}

int gemm_kernel_name(int ta, int tb, const GemmPlan &plan, char *name, size_t bytes)
{
    const bool small = plan.tile == T64_SMALL;
    const Shape &s = kShapes[small ? T64 : plan.tile];
    return snprintf(name, bytes, "gemm_direct_kernel<%s, %s, %d, %d, %d, %s, false>", ta ? "true" : "false", tb ? "true" : "false", s.bm, s.bn,
                    s.res, small ? "true" : "false");
}

int gemm_chain_kernel_name(const GemmPlan &plan, char *name, size_t bytes)
{
    const bool small = plan.tile == T64_SMALL;
    const Shape &s = kShapes[small ? T64 : plan.tile];
    return snprintf(name, bytes, "gemm_chain_kernel<%d, %d, %d, %s>", s.bm, s.bn, s.res, small ? "true" : "false");
}

// A program has few shapes and calls them over and over; working one out takes some microseconds (hundreds of costs), so
// each thread keeps the plans of the last ones by their sizes.
static GemmPlan kept_plan(int64_t M, int64_t N, int64_t K, int64_t nz, size_t lent, int chain)
{
    struct Kept {
        int64_t M, N, K, nz, how;                 // how: compute units and chain; 0: none kept
        size_t lent;
        GemmPlan plan;
    };
    static thread_local Kept kept[256] = {};
    const int64_t cus = device_cus(), how = cus * 8 + chain;
    const uint64_t h = ((uint64_t)M * 0x9e3779b97f4a7c15u ^ (uint64_t)N * 0xc2b2ae3d27d4eb4fu ^ (uint64_t)K * 0x165667b19e3779f9u) +
                       (uint64_t)(nz * 2 + (lent > 0 ? 1 : 0) + chain * 64) * 0x27d4eb2f165667c5u;
    Kept &k = kept[h >> 56];
    if (k.how != how || k.M != M || k.N != N || k.K != K || k.nz != nz || k.lent != lent)
        k = {M, N, K, nz, how, lent, make_plan(cus, M, N, K * chain, nz, lent, chain > 1 ? kChainShapes : kNumShapes)};
    return k.plan;
}
GemmPlan gemm_plan(int64_t M, int64_t N, int64_t K, int64_t nz, size_t lent) { return kept_plan(M, N, K, nz, lent, 1); }
GemmPlan gemm_plan_chain(int64_t M, int64_t N, int64_t K, int chain) { return kept_plan(M, N, K, 1, 0, chain); }

GemmPlan gemm_plan_parts(int64_t M, int64_t N, int64_t K, int parts)
{
    GemmPlan best = {-1, T64, 0, parts, 0};
    for (int t = T64; t < kNumShapes; t++) {
        const double c = has_parts(t) ? part_cost(device_cus(), t, M, N, (K + BK - 1) / BK, parts, 1.0) : -1.0;
        if (c >= 0 && (best.tile < 0 || c < best.us)) best = {t, T64, 0, parts, c};
    }
    return best;
}

// The same for operands that are loaded through registers whatever their alignment: 64 x 64 tiles, whose k tiles take some
// half longer than the direct ones' (64 x 128 and 128 x 128 took twice and three times as long as that: their loads have
// no room in the registers to be far enough ahead).
GemmPlan gemm_plan_any(int64_t M, int64_t N, int64_t K, size_t lent)
{
    const int64_t kt = (K + BK - 1) / BK, cus = device_cus();
    const double fixed = kShapes[T64].fixed;
    GemmPlan best = {T64, T64, 0, 1, 0};
    best.us = fixed + kAnyPerTile * (tile_cost(cus, T64, M, N, 1, kt) - fixed);
    split_k(cus, T64, M, N, kt, kAnyPerTile, best.us, lent, best);
    return best;
}

// What a launch of both is expected to take: the workgroups that the device holds at a time share them all, unless one of the
// longer product takes longer than that.  Separate launches -> one, us: S = 611, N = K = 1024 12.0 -> 8.7; three of those 23.7 ->
// 17.9; two of N = 2816 35.9 -> 28.4; 2048, 2048, 2048 41.4 -> 34.8; 333, 3200, 8640 61.7 -> 49.4; three of 128, 256, 256 (four
// launches) 16.3 -> 6.5.  Larger ones fill the device by themselves, with tiles of their own, and the long sums of the input
// gradient share their CUs with the other product's workgroups, which this estimate leaves out: two of 603, 9280, 3200 214 -> 246,
// two of 777, 8640, 3200 215 -> 233, 1351, 24104, 2048 292 -> 322.  So none beyond 150 us, where 49 products took 0.99 of the time
// apart in the mean and every third longer, and from 40 us on, where the tile costs are 2 to 3 us off, a gain of 8 % is asked for
// (1854, 2984, 3200 73 -> 80).  Of 2500 others (S 33 .. 2048, widths 256 .. 3200) 22 are 2 to 13 % slower as one, 59 us together
// (1961, 2672, 2048 53 -> 60; 80, 3200, 11120, bound by what it reads and writes, 49 -> 55); all of them 70.6 -> 59.2 ms.
GemmPlan gemm_plan_pair(int64_t S, int64_t N, int64_t K, int n, size_t lent)
{
    const int64_t cus = device_cus(), kt_nn = (N + BK - 1) / BK * n, kt_tn = (S + BK - 1) / BK;
    const bool small_nn = S * K <= kSmallOutput, small_tn = N * K <= kSmallOutput;
    GemmPlan best = {-1, T64, 0, 1, 0};
    if (small_nn != small_tn) return best;
    for (int tile : kPairShapes) {
        if ((tile == T64_SMALL) != small_nn) continue;
        const Shape &t = kShapes[tile == T64_SMALL ? T64 : tile];
        auto tiles = [&](int64_t M, int64_t C) { return (double)((M + t.bm - 1) / t.bm) * (double)((C + t.bn - 1) / t.bn); };
        const double work = tiles(S, K) * (kt_nn * t.full + t.round) + n * tiles(N, K) * (kt_tn * t.full + t.round);
        const double us = t.fixed + std::max(work / (double)(cus * t.res), (double)std::max(kt_nn, kt_tn) * (t.first + t.load));
        if (best.tile < 0 || us < best.us) {
            best.tile = tile;
            best.us = us;
        }
    }
    const GemmPlan nn = n > 1 ? gemm_plan_chain(S, K, N, n) : gemm_plan(S, K, N, 1, lent), tn = gemm_plan(N, K, S, n, 0);
    const double apart = nn.us + tn.us;
    if (apart > 150.0 || best.us >= (apart < 40.0 ? 0.95 : 0.92) * apart) best.tile = -1;
    return best;
}

int gemm_pair_launch(const GemmArgs &nn, const GemmArgs &tn, int64_t nblk, const GemmPlan &plan, hipStream_t st)
{
    const PairArgs p = {0, 0, nn, tn};
    switch (plan.tile) {
        case T64_SMALL: return launch_pair<T64_SMALL>(p, nblk, st);
        case 0: return launch_pair<0>(p, nblk, st);
        case 3: return launch_pair<3>(p, nblk, st);
        case 5: return launch_pair<5>(p, nblk, st);
        default: return launch_pair<7>(p, nblk, st);
    }
}

int gemm_direct_launch(int ta, int tb, const GemmArgs &p, int64_t nblk, const GemmPlan &plan, hipStream_t st)
{
    if (plan.split > 1) {
        GemmArgs q = p;
        q.split_tiles = (int)(((p.K + BK - 1) / BK + plan.split - 1) / plan.split);
        const int rc = launch_parts(ta, tb, plan.tile, q, plan.split, st);
        if (rc) return rc;
        const unsigned grid = (unsigned)((p.M * p.ldp + 1023) / 1024);
        const bool vec = p.N % 4 == 0 && p.ldc % 4 == 0 && aligned(p.C, 8);
        const auto reduce = plan.split <= 4 ? (vec ? reduce_parts_kernel<true, 4> : reduce_parts_kernel<false, 4>)
                                            : (vec ? reduce_parts_kernel<true, kMostParts> : reduce_parts_kernel<false, kMostParts>);
        hipLaunchKernelGGL(reduce, dim3(grid), dim3(256), 0, st, p.M, p.N, p.ldp, plan.split, p.part, p.alpha, p.beta, p.C, p.ldc);
        return launch_status("gemm_reduce_parts");
    }
    GemmArgs a = p;
    a.part = nullptr;
    if (plan.cols == 0) return launch_tile(ta, tb, plan.tile == T64_SMALL && p.odd ? T64 : plan.tile, a, nblk, st);
    GemmArgs b = a;
    a.N = plan.cols;
    b.N = p.N - a.N;
    b.B = p.B + (tb ? a.N * p.ldb : a.N);
    b.C = p.C + a.N;
    const int rc = launch_tile(ta, tb, plan.tile, a, nblk, st);
    return rc ? rc : launch_tile(ta, tb, plan.rest, b, nblk, st);
}

// a copy of up to two operands in the layout of the direct kernels (dst null: none of that one)
int gemm_repack(const half_t *const src[2], half_t *const dst[2], const int64_t rows[2], const int64_t cols[2], const int64_t ld[2],
                hipStream_t st)
{
    RepackArgs p;
    int64_t most = 0;
    for (int z = 0; z < 2; z++) {
        p.src[z] = src[z];
        p.dst[z] = dst[z];
        p.rows[z] = rows[z];
        p.cols[z] = cols[z];
        p.ld[z] = ld[z];
        if (dst[z]) most = std::max(most, rows[z] * ((cols[z] + 7) / 8));
    }
    CACTI_REQUIRE((most + 255) / 256 < (int64_t)1 << 31, CACTI_E_NOTIMPL, "gemm: operand too large to lay out");
    hipLaunchKernelGGL(repack_kernel, dim3((unsigned)((most + 255) / 256), 2), dim3(256), 0, st, p);
    return launch_status("gemm_repack");
}

}  // namespace cacti
