// Causal attention of short sequences, and of longer ones of few heads: the arithmetic and the rounding points of attention.hip
// on another split of the work.
//
// There a workgroup has 64 or 128 rows and its waves walk the keys together, a tile per step behind a barrier, each step 1.2 to
// 1.4 us of a chain (tile, product, exponentials, product) with nothing beside it: at 128 positions of 4 heads 9 us, of which
// the products are not one, and at 1000 positions of 4 heads 32 workgroups on 256 CUs.  Here a workgroup has 32 rows (keys, for
// dK and dV), four times as many workgroups, and its 4 or 8 waves split what is walked, block by block of 32: each wave loads
// its own blocks straight into its own LDS and waits for its own loads alone, so a walk is 1/4 or 1/8 as long and has no
// barrier, and the waves' sums meet in LDS once at the end.  The rounded scores stay in registers (forward), so that no product is
// formed twice: a wave sums its exponentials against its own keys' maximum, those sums are rescaled once, where the waves'
// statistics meet, and the probabilities are formed with the row's maximum and sum.
// Times, and where the lines between the two lie: at the bottom.
#include "attention_tile.h"

#include <algorithm>

namespace cacti {

namespace {

constexpr int kBlk = 32;                        // rows of a block: the fixed operand of a workgroup, a step of a wave
constexpr int kBlkB = kBlk * kRowB;             // 8 KB of LDS

// 32 x Dh of a [S, H, Dh] tensor straight into LDS by one wave (the layout of DmaTileMap, 4 rows per instruction)
struct BlockMap {
    int r0, pc;
    int64_t ld;
    int left;                                   // of the window: columns
    __device__ __forceinline__ BlockMap(int64_t ld_, int Dh, int shift) : ld(ld_), left(Dh + shift)
    {
        const int t = threadIdx.x & 63;
        pc = t & 15;
        r0 = t >> 4;
    }
    // instruction `it` of the 8; src = the window's first element in the block's first row; rows beyond the tensor are its last
    // row once more, so that a block is 8 loads to wait for whatever its rows (zero_rows where a product sums over them)
    __device__ __forceinline__ void load1(int it, gptr_t src, int rows, uint32_t lds) const
    {
        const int r = r0 + 4 * it, c = pc ^ gsw(r);
        if (c * 8 < left) dma16(lds + it * 4 * kRowB, (uint32_t)((min(r, rows - 1) * ld + c * 8) * 2), src);
    }
    __device__ __forceinline__ void load(gptr_t src, int rows, uint32_t lds) const
    {
#pragma unroll
        for (int it = 0; it < 8; it++) load1(it, src, rows, lds);
    }
};
constexpr int kPerBlock = 8;                    // instructions of a block's load

// The wave's own loads into LDS are waited for by the wave, but for the newest N; nothing of LDS is read ahead of it
template <int N>
__device__ __forceinline__ void landed()
{
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
// the wave's reads of LDS are through (what comes next may overwrite what they read)
__device__ __forceinline__ void reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

__device__ __forceinline__ uint32_t lds_of(const void *p) { return (uint32_t)(uintptr_t)p; }

// Rows [rows, 32) of a block that has landed, by its wave.  For the operand of a product over the block's rows whose other factor
// is 0 there: the last row is live for the queries (keys) that see it, and an infinity in it, once more times 0, would make
// their sums NaN.
__device__ __forceinline__ void zero_rows(unsigned char *block, int rows)
{
    for (int i = rows * 16 + (threadIdx.x & 63); i < kBlk * 16; i += 64) *reinterpret_cast<uint4 *>(block + i * 16) = make_uint4(0, 0, 0, 0);
}

// the chunks of a wave's blocks that no load writes
__device__ __forceinline__ void zero_block_pads(unsigned char *blocks, int rows, int nch)
{
    const int npad = 16 - nch;
    for (int i = threadIdx.x & 63; i < rows * npad; i += 64) {
        const int r = i / npad, c = nch + i % npad;
        *reinterpret_cast<uint4 *>(blocks + toff(r, c)) = make_uint4(0, 0, 0, 0);
    }
}

// Every wave's partial tile (DT x 16 floats per lane) is in its own part of LDS (`all`, per_wave bytes each); wave wid sums the
// groups of four columns that it answers for over the waves.  out(dt, q, sums): columns 32 dt + 8 q + 4 lh .. + 3 of row l32.
template <int DT, int NW, class F>
__device__ __forceinline__ void sum_partials(const unsigned char *all, int per_wave, int wid, int lane, F &&out)
{
    constexpr int GROUPS = DT * 4 / NW;
    static_assert(GROUPS >= 1, "a group of columns for every wave");
#pragma unroll
    for (int g = 0; g < GROUPS; g++) {
        const int grp = wid * GROUPS + g;
        float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const float *x = reinterpret_cast<const float *>(all + w * per_wave) + grp * 256 + lane;
#pragma unroll
            for (int r = 0; r < 4; r++) a[r] = w ? a[r] + x[r * 64] : x[r * 64];
        }
        out(grp >> 2, grp & 3, a);
    }
}
template <int DT>
__device__ __forceinline__ void put_partial(unsigned char *mine, const float16_t (&acc)[DT], int lane)
{
    float *x = reinterpret_cast<float *>(mine) + lane;
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) x[(dt * 16 + r) * 64] = acc[dt][r];
}
__device__ __forceinline__ void stage4(unsigned char *stage, int row, int dt, int q, int lh, const float (&a)[4], float scale)
{
    half4_t o;
#pragma unroll
    for (int r = 0; r < 4; r++) o[r] = f2h(scaled(scale, a[r]));
    *reinterpret_cast<half4_t *>(stage + toff(row, 4 * dt + q) + 8 * lh) = o;
}

constexpr size_t query_smem(int waves, bool adjoint)
{
    return (size_t)waves * 2 * kBlkB + (adjoint ? 3 : 1) * kBlkB + (size_t)waves * 2 * kBlk * sizeof(float);
}

// O and the statistics of 32 queries.  NW waves, at most NB key blocks of 32 for each.  With 8 waves and one workgroup per CU
// while there are no more workgroups than CUs, with 4 waves two per CU beyond: 1000 positions of 4 heads of 100 12.0 us with 8
// against 15.3 with 4, 640 of 32 of 100 21.4 against 16.4.
template <int KS, int DT, bool FAST, int NW, int NB>
__global__ void __launch_bounds__(NW * 64, 2) attn_short_fwd_kernel(AttnArgs p)
{
    asm volatile("" ::"s"(p.S), "s"(p.H), "s"(p.Dh), "s"(p.ld), "s"(p.alpha), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.out), "s"(p.m), "s"(p.l));
    typedef AttnMath<FAST> M;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *Qt = smem + NW * 2 * kBlkB;
    float *xs = reinterpret_cast<float *>(Qt + kBlkB);                   // [NW][2][32]
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, lh = lane >> 5;
    unsigned char *mine = smem + wid * 2 * kBlkB;
    const int S = p.S, Dh = p.Dh;
    const int64_t ld = p.ld;
    const int nq = (S + kBlk - 1) / kBlk, h = blockIdx.x % p.H, qt = nq - 1 - blockIdx.x / p.H;
    const int shift = (int)(((int64_t)h * Dh) & 7), i0 = qt * kBlk, myrow = i0 + l32;
    const int64_t hoff = (int64_t)h * Dh - shift;
    const BlockMap bm(ld, Dh, shift);
    // key blocks wid, wid + NW, ..; load s of the wave is key block s, then (s >= n) value block s - n, in buffer s & 1
    const int n = wid <= qt ? (qt - wid) / NW + 1 : 0;
    auto issue = [&](int s) __attribute__((always_inline)) {
        const int kb = wid + NW * (s < n ? s : s - n);
        bm.load((s < n ? gp(p.k) : gp(p.v)) + hoff + (int64_t)kb * kBlk * ld, min(S - kb * kBlk, kBlk), lds_of(mine + (s & 1) * kBlkB));
    };
#pragma unroll
    for (int i = 0; i < 8 / NW; i++) bm.load1(wid * (8 / NW) + i, gp(p.q) + hoff + (int64_t)i0 * ld, min(S - i0, kBlk), lds_of(Qt));
    if (n > 0) {
        issue(0);
        issue(1);
    }
    zero_block_pads(mine, 2 * kBlk, (Dh + shift + 7) >> 3);
    if (n > 0) landed<2 * kPerBlock>();
    else landed<0>();
    __syncthreads();
    half8_t qf[KS];
    frags_from_tile<KS>(qf, Qt, l32, Dh, lh, shift);

    // scores of all of the wave's blocks, rounded, in registers
    half2v_t sc[NB][8];
    const half_t ninf = (half_t)-INFINITY;
    half2v_t mx = {ninf, ninf};
    static_for<0, NB>([&](auto j_c) __attribute__((always_inline)) {
        constexpr int j = decltype(j_c)::value;
        if (j < n) {
            landed<kPerBlock>();
            const float16_t acc = prod_direct<KS>(mine + (j & 1) * kBlkB, 0, qf, l32, lh);
            reads_done();
            if (n > 1) issue(j + 2);
            const int kb = wid + NW * j;
            if (kb < qt) {
#pragma unroll
                for (int e = 0; e < 8; e++) sc[j][e] = half2v_t{f2h(scaled(p.alpha, acc[2 * e])), f2h(scaled(p.alpha, acc[2 * e + 1]))};
            } else {
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int key = kb * kBlk + 8 * (e >> 2) + 4 * lh + (e & 3);
                    sc[j][e >> 1][e & 1] = key <= myrow ? f2h(scaled(p.alpha, acc[e])) : ninf;
                }
            }
#pragma unroll
            for (int e = 0; e < 8; e++) mx = __builtin_elementwise_max(mx, sc[j][e]);
        }
    });
    // the row's maximum and sum over the wave's keys, then over the waves
    float m = (float)__builtin_fmaxf16(mx[0], mx[1]), l = 0.f;
    m = with32(m, OpMax());
    const float c = m * kLog2e;
    static_for<0, NB>([&](auto j_c) __attribute__((always_inline)) {
        constexpr int j = decltype(j_c)::value;
        if (j < n) {
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const half_t s = sc[j][e >> 1][e & 1];
                l += s == ninf ? 0.f : FAST ? exp2_mix(s, c) : M::ex((float)s, m);
            }
        }
    });
    l = with32(l, OpSum());
    if (lh == 0) {
        xs[(wid * 2 + 0) * kBlk + l32] = m;
        xs[(wid * 2 + 1) * kBlk + l32] = l;
    }
    __syncthreads();
    m = xs[l32];
#pragma unroll
    for (int w = 1; w < NW; w++) m = fmaxf(m, xs[w * 2 * kBlk + l32]);
    l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const float mw = xs[w * 2 * kBlk + l32], lw = xs[(w * 2 + 1) * kBlk + l32];
        l += mw == -INFINITY ? lw : lw * M::ex(mw, m);       // (0 then, or NaN of scores that are NaN)
    }
    if (myrow >= S) {
        m = 0.f;
        l = 1.f;
    } else if (wid == 0 && lh == 0) {
        p.m[(int64_t)h * S + myrow] = m;
        p.l[(int64_t)h * S + myrow] = l;
    }
    const float y = recip_refined(l), cs = prob_shift(m, l);

    const bool ragged = S - i0 < kBlk && (qt - wid) % NW == 0;      // the wave's last value block
    float16_t oacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[dt][r] = 0.f;
    static_for<0, NB>([&](auto j_c) __attribute__((always_inline)) {
        constexpr int j = decltype(j_c)::value;
        if (j < n) {
            float pe[16];
            // masked by position: a row whose every score came to -infinity has no probabilities (NaN), 0 is for the keys behind it
            const int last = wid + NW * j < qt ? kBlk : l32 - 4 * lh;
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const half_t s = sc[j][e >> 1][e & 1];
                pe[e] = FAST ? exp2_mix(s, cs) : 8 * (e >> 2) + (e & 3) <= last ? M::prob((float)s, m, l, y) : 0.f;
            }
            const half8_t y0 = pack8(pe), y1 = pack8(pe + 8);
            if (j + 1 < n) {
                landed<kPerBlock>();
            } else {
                landed<0>();
                if (ragged) zero_rows(mine + ((n + j) & 1) * kBlkB, S - i0);
            }
            prod_tr<DT>(oacc, mine + ((n + j) & 1) * kBlkB, 0, y0, y1, lane);
            if (j + 2 < n) {
                reads_done();
                issue(n + j + 2);
            }
        }
    });
    reads_done();
    put_partial<DT>(mine, oacc, lane);
    __syncthreads();
    sum_partials<DT, NW>(smem, 2 * kBlkB, wid, lane, [&](int dt, int q, const float (&a)[4]) { stage4(Qt, l32, dt, q, lh, a, 1.0f); });
    __syncthreads();
    write_rows<kBlk>(Qt, p.out + (int64_t)i0 * ld + hoff, ld, min(kBlk, S - i0), Dh, shift, threadIdx.x, NW * 64);
}

// dQ of 32 queries, and the rows' offsets y and sigmas for the dK / dV kernel, whichever that is.  8 waves: 4 are slower from
// 300 positions on (611, 16 of 64 15.0 us against 14.3; 1000, 4 of 100 14.6 against 12.7).
template <int KS, int DT, bool FAST>
__global__ void __launch_bounds__(512, 2) attn_short_dq_kernel(AttnArgs p)
{
    constexpr int NW = 8;
    asm volatile("" ::"s"(p.S), "s"(p.H), "s"(p.Dh), "s"(p.ld), "s"(p.alpha), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.dO), "s"(p.o), "s"(p.dq),
                 "s"(p.m), "s"(p.l), "s"(p.y), "s"(p.sig), "s"(p.acc_dq));
    typedef AttnMath<FAST> M;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *Qt = smem + NW * 2 * kBlkB, *Gt = Qt + kBlkB, *Ot = Gt + kBlkB;
    float *xs = reinterpret_cast<float *>(Ot + kBlkB);                   // [NW][32]
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, lh = lane >> 5;
    unsigned char *Ks = smem + wid * 2 * kBlkB, *Vs = Ks + kBlkB;
    const int S = p.S, Dh = p.Dh;
    const int64_t ld = p.ld;
    const int nq = (S + kBlk - 1) / kBlk, h = blockIdx.x % p.H, qt = nq - 1 - blockIdx.x / p.H;
    const int shift = (int)(((int64_t)h * Dh) & 7), i0 = qt * kBlk, myrow = i0 + l32;
    const int64_t hoff = (int64_t)h * Dh - shift;
    // this lane's row, and the one it votes for on the form of sigma
    gfptr_t lrow = (gfptr_t)p.l + (int64_t)h * S;
    const int vrow = (i0 & ~127) + (threadIdx.x & 127);
    float m = ((gfptr_t)p.m)[(int64_t)h * S + min(myrow, S - 1)], l = lrow[min(myrow, S - 1)];
    const float lvote = lrow[min(vrow, S - 1)];
    const BlockMap bm(ld, Dh, shift);
    // key blocks wid, wid + NW, ..
    const int n = wid <= qt ? (qt - wid) / NW + 1 : 0;
    auto issue = [&](const half_t *X, unsigned char *to, int j) __attribute__((always_inline)) {
        const int kb = wid + NW * j;
        bm.load(gp(X) + hoff + (int64_t)kb * kBlk * ld, min(S - kb * kBlk, kBlk), lds_of(to));
    };
    const bool want_o = FAST && p.o;
#pragma unroll
    for (int i = 0; i < 8 / NW; i++) {
        const int it = wid * (8 / NW) + i, rows = min(S - i0, kBlk);
        const int64_t off = hoff + (int64_t)i0 * ld;
        bm.load1(it, gp(p.q) + off, rows, lds_of(Qt));
        bm.load1(it, gp(p.dO) + off, rows, lds_of(Gt));
        if (want_o) bm.load1(it, gp(p.o) + off, rows, lds_of(Ot));
    }
    if (n > 0) {
        issue(p.v, Vs, 0);
        issue(p.k, Ks, 0);
    }
    zero_block_pads(Ks, 2 * kBlk, (Dh + shift + 7) >> 3);
    if (n > 0) landed<2 * kPerBlock>();
    else landed<0>();
    // (which form of sigma: attn_bwd_dq_kernel)
    const bool short_sigma = __syncthreads_and(want_o && (vrow >= S || lvote >= kSpread)) != 0;
    if (myrow >= S) {
        m = 0.f;
        l = 1.f;
    }
    const float y = recip_refined(l), cs = prob_shift(m, l);
    half8_t qf[KS], gf[KS];
    frags_from_tile<KS>(qf, Qt, l32, Dh, lh, shift);
    frags_from_tile<KS>(gf, Gt, l32, Dh, lh, shift);

    float sig = 0.f;
    float16_t dacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) dacc[dt][r] = 0.f;
    // Over the wave's key blocks, the first of which is on its way.  The values are used up before the keys are, so the next
    // ones take their place while the block's arithmetic runs.
    auto run_pass = [&](auto pass_c) __attribute__((always_inline)) {
        constexpr int PASS = decltype(pass_c)::value;
        float part = 0.f;
#pragma unroll 1
        for (int j = 0; j < n; j++) {
            landed<kPerBlock>();
            const float16_t pacc = prod_direct<KS>(Vs, 0, gf, l32, lh);
            reads_done();
            if (j + 1 < n) {
                issue(p.v, Vs, j + 1);
                landed<kPerBlock>();
            } else {
                landed<0>();
            }
            const float16_t sacc = prod_direct<KS>(Ks, 0, qf, l32, lh);
            const int kb = wid + NW * j;
            float de[16];
            auto elems = [&](auto full_c) __attribute__((always_inline)) {
                constexpr bool FULL = decltype(full_c)::value;
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const bool live = FULL || kb * kBlk + 8 * (e >> 2) + 4 * lh + (e & 3) <= myrow;
                    const half_t d = f2h(pacc[e]);
                    if constexpr (FAST) {
                        const float pr = exp2_mix(f2h(scaled(p.alpha, sacc[e])), cs);
                        if (PASS == 0) part = live ? __builtin_fmaf((float)d, pr, part) : part;
                        else de[e] = live ? __builtin_fmaf((float)d, pr, -(sig * pr)) : 0.f;
                    } else {
                        const float pr = M::prob(rnd16(scaled(p.alpha, sacc[e])), m, l, y), t = pr * (float)d;
                        if (PASS == 0) part += live ? t : 0.f;
                        else de[e] = live ? t - sig * pr : 0.f;
                    }
                }
            };
            if (kb < qt) elems(std::true_type{});        // no masks on blocks wholly below the diagonal
            else elems(std::false_type{});
            if (PASS == 1) prod_tr<DT>(dacc, Ks, 0, pack8(de), pack8(de + 8), lane);
            reads_done();
            if (j + 1 < n) issue(p.k, Ks, j + 1);
        }
        return part;
    };
    if (short_sigma) {
        half8_t of[KS];
        frags_from_tile<KS>(of, Ot, l32, Dh, lh, shift);
        float part = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int e = 0; e < 8; e++) part = __builtin_fmaf((float)gf[ks][e], (float)of[ks][e], part);
        sig = with32(part, OpSum());
    } else {
        float part = run_pass(std::integral_constant<int, 0>{});
        if (n > 0) {
            issue(p.v, Vs, 0);
            issue(p.k, Ks, 0);
        }
        part = with32(part, OpSum());
        if (lh == 0) xs[wid * kBlk + l32] = part;
        __syncthreads();
        sig = xs[l32];
#pragma unroll
        for (int w = 1; w < NW; w++) sig += xs[w * kBlk + l32];
    }
    if (wid == 0 && lh == 0 && myrow < S) {
        p.y[(int64_t)h * S + myrow] = FAST ? cs : y;
        p.sig[(int64_t)h * S + myrow] = sig;
    }
    run_pass(std::integral_constant<int, 1>{});
    put_partial<DT>(Ks, dacc, lane);
    __syncthreads();
    sum_partials<DT, NW>(smem, 2 * kBlkB, wid, lane, [&](int dt, int q, const float (&a)[4]) {
        if (!p.acc_dq) {
            stage4(Qt, l32, dt, q, lh, a, p.alpha);
        } else {
            const int d0 = 32 * dt + 8 * q + 4 * lh - shift;
            if (myrow < S && d0 >= 0 && d0 < Dh)
                store_row4(p.dq + (int64_t)myrow * ld + (int64_t)h * Dh + d0, a[0], a[1], a[2], a[3], p.alpha, 1);
        }
    });
    if (!p.acc_dq) {
        __syncthreads();
        write_rows<kBlk>(Qt, p.dq + (int64_t)i0 * ld + hoff, ld, min(kBlk, S - i0), Dh, shift, threadIdx.x, NW * 64);
    }
}

// dK and dV of 32 keys.  8 waves of one pair of blocks (queries, dO) each with heads to 64 (300 positions of 8 8.2 us, against
// 10.5 with 4 waves); the two sums of wider heads are 128 registers, which 4 waves have room for (1024, 16 of 128 28.9 us against
// 45.4 with 8, which spill), with a second pair on its way.
constexpr int key_waves(int dt) { return dt == 2 ? 8 : 4; }
constexpr size_t kKeySmem = 8 * 2 * kBlkB + 2 * kBlkB + 8 * 4 * 64 * sizeof(float);       // with 8 waves of one pair, 4 of two

template <int KS, int DT, bool FAST>
__global__ void __launch_bounds__(key_waves(DT) * 64, key_waves(DT) / 4) attn_short_dkv_kernel(AttnArgs p)
{
    asm volatile("" ::"s"(p.S), "s"(p.H), "s"(p.Dh), "s"(p.ld), "s"(p.alpha), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.dO), "s"(p.dk), "s"(p.dv),
                 "s"(p.m), "s"(p.l), "s"(p.y), "s"(p.sig), "s"(p.acc_dk), "s"(p.acc_dv));
    typedef AttnMath<FAST> M;
    constexpr int NW = key_waves(DT), PAIRS = 8 / NW, kWaveB = PAIRS * 2 * kBlkB, NST = FAST ? 2 : 4, PAIR = 2 * kPerBlock + NST;
    static_assert(2 * DT * 4096 <= kWaveB, "a wave's blocks hold its partial tiles of dK and dV");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *Kt = smem + NW * kWaveB, *Vt = Kt + kBlkB;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, lh = lane >> 5;
    unsigned char *mine = smem + wid * kWaveB;
    float *st = reinterpret_cast<float *>(Vt + kBlkB) + wid * PAIRS * 4 * 64;    // [PAIRS][y, sigma, m, l][64]
    const int S = p.S, Dh = p.Dh;
    const int64_t ld = p.ld;
    const int nq = (S + kBlk - 1) / kBlk, h = blockIdx.x % p.H, kt = blockIdx.x / p.H;
    const int shift = (int)(((int64_t)h * Dh) & 7), c0 = kt * kBlk, mykey = c0 + l32;
    const int64_t hoff = (int64_t)h * Dh - shift;
    const BlockMap bm(ld, Dh, shift);
    // query blocks kt + wid, + NW, ..
    const int n = kt + wid < nq ? (nq - 1 - kt - wid) / NW + 1 : 0;
    gfptr_t stats[4] = {(gfptr_t)p.y + (int64_t)h * S, (gfptr_t)p.sig + (int64_t)h * S, (gfptr_t)p.m + (int64_t)h * S, (gfptr_t)p.l + (int64_t)h * S};
    auto issue_q = [&](int j) __attribute__((always_inline)) {
        const int q0 = (kt + wid + NW * j) * kBlk;
        bm.load(gp(p.q) + hoff + (int64_t)q0 * ld, min(S - q0, kBlk), lds_of(mine + j % PAIRS * 2 * kBlkB));
    };
    auto issue_g = [&](int j) __attribute__((always_inline)) {           // dO and the rows' statistics
        const int q0 = (kt + wid + NW * j) * kBlk;
        bm.load(gp(p.dO) + hoff + (int64_t)q0 * ld, min(S - q0, kBlk), lds_of(mine + j % PAIRS * 2 * kBlkB + kBlkB));
#pragma unroll
        for (int a = 0; a < NST; a++) {
            const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds_of(st + (j % PAIRS * 4 + a) * 64));
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                         :
                         : "s"(m0), "v"((uint32_t)min(q0 + lane, S - 1) * 4u), "s"(stats[a])
                         : "memory");
        }
    };
#pragma unroll
    for (int i = 0; i < 8 / NW; i++) {
        bm.load1(wid * (8 / NW) + i, gp(p.k) + hoff + (int64_t)c0 * ld, min(S - c0, kBlk), lds_of(Kt));
        bm.load1(wid * (8 / NW) + i, gp(p.v) + hoff + (int64_t)c0 * ld, min(S - c0, kBlk), lds_of(Vt));
    }
    if (n > 0) {
        issue_g(0);
        issue_q(0);
    }
    zero_block_pads(mine, PAIRS * 2 * kBlk, (Dh + shift + 7) >> 3);
    if (n > 0) landed<PAIR>();
    else landed<0>();
    __syncthreads();
    half8_t kf[KS], vf[KS];
    frags_from_tile<KS>(kf, Kt, l32, Dh, lh, shift);
    frags_from_tile<KS>(vf, Vt, l32, Dh, lh, shift);
    float16_t kacc[DT], vacc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            kacc[dt][r] = 0.f;
            vacc[dt][r] = 0.f;
        }
    if (PAIRS == 2 && n > 1) {
        issue_g(1);
        issue_q(1);
    }
#pragma unroll 1
    for (int j = 0; j < n; j++) {
        if (PAIRS == 1) landed<kPerBlock>();
        else if (j + 1 < n) landed<PAIR>();
        else landed<0>();
        const unsigned char *Qs = mine + j % PAIRS * 2 * kBlkB, *Gs = Qs + kBlkB;
        const float *stc = st + j % PAIRS * 4 * 64;
        const int q0 = (kt + wid + NW * j) * kBlk;
        if (S - q0 < kBlk) zero_rows(mine + j % PAIRS * 2 * kBlkB + kBlkB, S - q0);
        const float16_t pacc = prod_direct<KS, NW == 8>(Gs, 0, vf, l32, lh);
        if (PAIRS == 1) landed<0>();
        const float16_t sacc = prod_direct<KS, NW == 8>(Qs, 0, kf, l32, lh);
        const bool full = q0 > c0 && q0 + kBlk <= S;
        float pe[16], de[16];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int qi = 8 * q + 4 * lh;
            const float4_t yy = *reinterpret_cast<const float4_t *>(stc + qi), sg = *reinterpret_cast<const float4_t *>(stc + 64 + qi);
            float4_t mm, ll;
            if constexpr (!FAST) {
                mm = *reinterpret_cast<const float4_t *>(stc + 128 + qi);
                ll = *reinterpret_cast<const float4_t *>(stc + 192 + qi);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int e = 4 * q + r, query = q0 + qi + r;
                const half_t d = f2h(pacc[e]);
                float pr, ds;
                if constexpr (FAST) {
                    pr = exp2_mix(f2h(scaled(p.alpha, sacc[e])), yy[r]);
                    ds = __builtin_fmaf((float)d, pr, -(sg[r] * pr));
                } else {
                    pr = M::prob(rnd16(scaled(p.alpha, sacc[e])), mm[r], ll[r], yy[r]);
                    ds = pr * (float)d - sg[r] * pr;
                }
                const bool live = full || (query >= mykey && query < S);
                pe[e] = live ? pr : 0.f;
                de[e] = live ? ds : 0.f;
            }
        }
        prod_tr<DT>(vacc, Gs, 0, pack8(pe), pack8(pe + 8), lane);
        if (PAIRS == 1 && j + 1 < n) {
            reads_done();
            issue_g(j + 1);
        }
        prod_tr<DT>(kacc, Qs, 0, pack8(de), pack8(de + 8), lane);
        if (j + PAIRS < n) {
            reads_done();
            if (PAIRS == 2) issue_g(j + 2);
            issue_q(j + PAIRS);
        }
    }
    reads_done();
    put_partial<DT>(mine, kacc, lane);
    put_partial<DT>(mine + DT * 4096, vacc, lane);
    __syncthreads();
    auto out = [&](half_t *dst, unsigned char *stage, float scale, int acc) __attribute__((always_inline)) {
        return [=](int dt, int q, const float (&a)[4]) __attribute__((always_inline)) {
            if (!acc) {
                stage4(stage, l32, dt, q, lh, a, scale);
            } else {
                const int d0 = 32 * dt + 8 * q + 4 * lh - shift;
                if (mykey < S && d0 >= 0 && d0 < Dh)
                    store_row4(dst + (int64_t)mykey * ld + (int64_t)h * Dh + d0, a[0], a[1], a[2], a[3], scale, 1);
            }
        };
    };
    sum_partials<DT, NW>(smem, kWaveB, wid, lane, out(p.dk, Kt, p.alpha, p.acc_dk));
    sum_partials<DT, NW>(smem + DT * 4096, kWaveB, wid, lane, out(p.dv, Vt, 1.0f, p.acc_dv));
    __syncthreads();
    const int64_t off = (int64_t)c0 * ld + hoff;
    if (!p.acc_dk) write_rows<kBlk>(Kt, p.dk + off, ld, min(kBlk, S - c0), Dh, shift, threadIdx.x, NW * 64);
    if (!p.acc_dv) write_rows<kBlk>(Vt, p.dv + off, ld, min(kBlk, S - c0), Dh, shift, threadIdx.x, NW * 64);
}

int64_t blocks(int64_t S) { return (S + kBlk - 1) / kBlk; }

template <class K>
int launch(K kern, DeviceOnce &ready, size_t smem, int waves, const AttnArgs &p, hipStream_t st, const char *what)
{
    if (!ready.fresh()) {
        CACTI_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        ready.mark();
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(blocks(p.S) * p.H)), dim3(waves * 64), smem, st, p);
    return launch_status(what);
}

template <int KS, int DT, bool FAST, int NW, int NB>
int fwd_as(const AttnArgs &p, hipStream_t st)
{
    static DeviceOnce ready;
    return launch(attn_short_fwd_kernel<KS, DT, FAST, NW, NB>, ready, query_smem(NW, false), NW, p, st, "attention_fwd");
}
template <int KS, int DT, bool FAST> struct Fwd {
    static int run(const AttnArgs &p, hipStream_t st)
    {
        if (p.S > 1024) return fwd_as<KS, DT, FAST, 8, 8>(p, st);
        return blocks(p.S) * p.H > device_cus() ? fwd_as<KS, DT, FAST, 4, 8>(p, st) : fwd_as<KS, DT, FAST, 8, 4>(p, st);
    }
};
template <int KS, int DT, bool FAST> struct Dq {
    static int run(const AttnArgs &p, hipStream_t st)
    {
        static DeviceOnce ready;
        return launch(attn_short_dq_kernel<KS, DT, FAST>, ready, query_smem(8, true), 8, p, st, "attention_bwd_dq");
    }
};
template <int KS, int DT, bool FAST> struct Dkv {
    static int run(const AttnArgs &p, hipStream_t st)
    {
        static DeviceOnce ready;
        return launch(attn_short_dkv_kernel<KS, DT, FAST>, ready, kKeySmem, key_waves(DT), p, st, "attention_bwd_dkv");
    }
};
// the instantiation by the window span (16 KS and 32 DT positions cover it) and the arithmetic
template <template <int, int, bool> class L>
int dispatch(const AttnArgs &p, int64_t span, bool exact, hipStream_t st)
{
    if (span <= 64) return exact ? L<4, 2, false>::run(p, st) : L<4, 2, true>::run(p, st);
    if (span <= 112) return exact ? L<7, 4, false>::run(p, st) : L<7, 4, true>::run(p, st);
    return exact ? L<8, 4, false>::run(p, st) : L<8, 4, true>::run(p, st);
}

}  // namespace

// A workgroup of these kernels takes 32 rows, so each reads a head's keys (or queries) for a quarter of the rows that one of
// attention.hip reads them for: with many workgroups per CU that traffic is what they take, and the larger tiles are better.
// Where the lines lie, kernel times in us, attention.hip -> here, workgroups of 32 rows in brackets, 256 CUs:
//   forward, to 1024 positions: 128 positions of 4 heads of 64 (16) 8.9 -> 5.9; 1000, 4 of 100 (128) 23.0 -> 12.0; 512, 16 of
//   100 (256) 15.8 -> 9.7; 1024, 16 of 128 (512) 25.2 -> 17.5; 1000, 24 of 64 (768) 24.0 -> 20.5; 1024, 32 of 128 (1024) 30.6 ->
//   25.8; 512, 64 of 64 (1024) 16.7 -> 17.1; 1024, 64 of 64 (2048) 34.9 -> 41.6.  To 2048: 1536, 4 of 128 (192) 30.4 -> 15.3;
//   2048, 8 of 64 (512) 33.6 -> 23.4; 1531, 16 of 128 (768) 34.6 -> 32.9; 2048, 16 of 64 (1024) 40.7 -> 43.2.  Beyond 2048 the
//   rounded scores of a wave's blocks have no room in its registers.
//   The adjoint's workgroups have a CU to themselves, so beyond 256 they come in two rounds, and the second is worth it where the
//   first one's walks are long (second_round): up to 256 0.54 to 0.90 of the time.
//   dQ, break-even at 280 workgroups of 500 positions, 320 of 600, 360 of 700, 440 of 800 and 512 of 930: 128, 4 of 64 10.8 -> 7.4;
//   3001, 2 of 128 (188) 43.6 -> 25.0; 289, 27 of 64 (270) 10.8 -> 13.5; 373, 29 of 128 (348) 12.8 -> 15.6; 504, 26 of 64 (416) 12.7 ->
//   15.4; 593, 25 of 128 (475) 17.5 -> 20.4; on the other side 611, 16 of 64 (320) 1.00 of the time, 640 to 700 (257 .. 280) 0.93, 750 to
//   800 (to 340) 0.90 to 0.97, 800 to 900 (to 400) 0.82 to 0.96; 4096, 4 of 64 (512) 43.7 -> 37.3; 640, 32 of 100 (640) 23.0 -> 26.0;
//   1531, 16 of 128 (768) 34.5 -> 36.1.  Exact, where arithmetic takes more of a block: at 257 of 100 and 512 of 530 (168, 67 of 64 (402)
//   12.4 -> 15.2; 64 to 200 (257 .. 512) 1.03 to 1.11, 200 to 300 (to 350) 0.96, 300 to 400 (to 450) 0.80 to 0.97).
//   dK, dV, parts and their sum together, at 257 of 200 and 512 of 630: 128, 4 of 64 10.1 -> 6.2; 777, 16 of 128 (400) 26.4 -> 21.3;
//   1024, 16 of 64 (512) 27.6 -> 19.3; 2048, 8 of 128 (512) 46.7 -> 41.3; 168, 67 of 64 (402) 9.8 -> 13.0; 64 to 200 (257 .. 450) 1.07 to
//   1.17, 200 to 300 (to 400) 1.01 to 1.05, 300 to 400 (to 350) 0.86, 500 to 600 (to 450) 0.75 to 0.98, from there to 512 1.01; 1000, 24
//   of 64 (768) 23.5 -> 27.3; 640, 32 of 100 (640) 22.5 -> 30.4.
//   Exact arithmetic, (512): 512, 32 of 128 18.7 -> 15.0 forward; 2048, 8 of 64 47.0 -> 34.5, adjoint 106.7 -> 74.1.
bool attention_short_fwd_takes(int64_t S, int64_t H, int64_t span)
{
    const int64_t wgs = blocks(S) * H, cus = device_cus();
    return S <= 1024 ? wgs <= (span > 64 ? 4 : 3) * cus : S <= 2048 && wgs <= 2 * cus;
}
// The second round of workgroups: as many as the positions beyond `from` are 1/430 of the CUs'.
static bool second_round(int64_t S, int64_t H, int64_t from)
{
    const int64_t wgs = blocks(S) * H, cus = device_cus();
    return wgs <= cus || (wgs <= 2 * cus && (wgs - cus) * 430 <= (S - from) * cus);
}
bool attention_short_dq_takes(int64_t S, int64_t H, bool exact) { return second_round(S, H, exact ? 100 : 500); }

// Against the parts of attention.hip (`per` tiles of 64 queries each; 0: there are none): a wave's walk is blocks / waves long, at
// 1.7 us each, a part's `per` at 1.5 behind a longer start and the sum's launch.  Workgroups there -> here, us: 1000, 4 of 100
// (2 tiles, 8 blocks) 21.1 -> 20.2; 2048, 2 of 128 (4, 16) 26.5 -> 33.4; 2048, 4 of 128 (8, 16) 32.8 -> 34.3; 4096, 1 of 64 (8,
// 16) 26.3 -> 32.6; 4096, 2 of 64 (16, 16) 37.8 -> 34.2; 4096, 2 of 128 (16, 32) 51.3 -> 65.2.
bool attention_short_dkv_takes(int64_t S, int64_t H, int64_t span, int per)
{
    const int waves = span <= 64 ? 8 : 4;
    return second_round(S, H, 200) && (per == 0 || (blocks(S) + waves - 1) / waves <= per + 6);
}

int attention_short_fwd(const AttnArgs &p, int64_t span, bool exact, hipStream_t st) { return dispatch<Fwd>(p, span, exact, st); }
int attention_short_dq(const AttnArgs &p, int64_t span, bool exact, hipStream_t st) { return dispatch<Dq>(p, span, exact, st); }
int attention_short_dkv(const AttnArgs &p, int64_t span, bool exact, hipStream_t st) { return dispatch<Dkv>(p, span, exact, st); }

}  // namespace cacti
