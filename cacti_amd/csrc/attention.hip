// Causal attention of one layer as fused kernels: the reference's chain
//   S16 = f16(a Q K^T) -> f32 -> causal mask -> softmax -> P16 = f16(P) -> O = f16(P16 V)
// (src/librarium/llama.rs:501-507; BlockMatrixMul src/thunk/op.rs:4719-5471, BlockTriElemAffine
// :4189-4278, InnerSoftmax :3257-3383) and its adjoint
//   dV = f16(P16^T dO), dP16 = f16(dO V^T), dS16 = f16(tril(T - (sum_j T) P')), T = P' f32(dP16),
//   dQ = f16(a dS16 K), dK = f16(a dS16^T Q)
// (pop_adj :4882-4912, InnerSoftmaxPostAdj :3386-3457) without the sequence x sequence tensors
// ever reaching memory.  Every rounding point of the chain is kept, in registers: scores and
// probabilities are rounded to f16 before they are used, each product accumulates in fp32 and is
// rounded once.
//
// Layout: q, k, v, o and their adjoints are [S, H, Dh] (row stride ld), 8-byte aligned.
//
// Forward (a workgroup = 128 or 64 query rows of one head, 32 rows to a wave; keys in tiles of 64):
// the scores are computed twice.  Pass 1 keeps a running row maximum m and sum l of exp(S16 - m);
// pass 2 recomputes S16 (same instructions, same bits), forms P16 = f16(exp(S16 - m) / l) -- the
// reference's probabilities, not an unnormalised stand-in -- and accumulates O += P16 V.  Only
// (m, l) per row are kept for the adjoint.
//
// Adjoint: two kernels, each deterministic (no atomics).  The dQ kernel has the forward's shape
// (queries fixed, loop over keys); the dK/dV kernel fixes 128 or 64 keys and loops over the queries at
// or after them.  Both recompute S16, P' and dP16 per tile.  The row sums sigma_i = sum_j P'_ij
// f32(dP16_ij) are formed as the reference forms them, from the rounded dP16, by a first pass of the
// dQ kernel over its key tiles, unless the probability of every row of a block of 128 queries is spread
// (kSpread): the shortcut sum_d dO_id O_id is the same number only in exact arithmetic, and misses the
// cancellation between dP16 and sigma in rows whose probability sits on one key, where the reference's
// dS is exactly zero.
//
// MFMA data flow (v_mfma_f32_32x32x16_f16, D = X Y^T: lane <-> row of Y, registers <-> rows of X).
// With the fixed operand as Y, a lane owns one query (key) and 16 of a 32-key (query) tile's
// entries, 4 q + r <-> index 8 q + 4 lh + r.  Rounded to f16 and packed, registers 8 kk .. 8 kk + 7
// are directly the Y operand of k step kk of the next product (contraction over that index); the
// X operand is read from the [row][d] LDS tile by ds_read_b64_tr_b16 with the matching row
// permutation (rows 16 kk + 4 lh + 0..3 and 16 kk + 8 + 4 lh + 0..3).  No probability ever goes
// through LDS.
//
// LDS tiles are [rows][128 halves] (256 bytes per row = one pass over all 64 banks, head dim
// zero-padded); 16-byte chunk c of row r sits at chunk c ^ g(r), g(r) = 2 (r & 3) | ((r >> 2) & 1) |
// 8 (((r >> 3) ^ r) & 1): a permutation of r mod 16, so the 16-byte operand reads of 16 consecutive rows
// cover all 16 bank groups, and the 8 rows of a transposing read (64 bytes each out of one aligned
// 64-byte quarter of the row) fall two to a quarter, which is all 64 banks twice -- the least 512 bytes
// can take.  (With bit 3 of g taken from bit 3 of r alone those 8 rows shared two quarters: a quarter of
// all LDS cycles were bank conflicts then, 4 % now.)
//
// How a K / V (Q / dO) tile gets there: straight from memory by global_load_lds_dwordx4 where the tensors
// allow it (16-byte aligned, see DmaTileMap: every head addressed from the 16-byte boundary at or below
// its start), else through registers (FastTileLoader, TileLoader8).  Measured at 32 heads x 2048 x 100:
// forward 108.7 -> 92.9 us, adjoint 235.5 -> 209.8 us, 48 vector registers fewer per kernel.  On that path the
// fixed operand of a workgroup (its 128 rows) arrives as tiles in LDS as well and every wave picks its fragments
// out of them (frags_from_tile), and the outputs leave through LDS as whole row segments (stage_rows,
// write_rows): a load or store in which every lane addresses its own row costs about a clock per lane.
// Forward 85.9 -> 79.0 us, dQ 95.8 -> 84.8, dK / dV 101.9 -> 97.0.
#include "attention_tile.h"

#include <algorithm>
#include <atomic>
#include <initializer_list>

using namespace cacti;

namespace {

// Work split of the query-major kernels (forward, dQ).  A workgroup is two wave groups of 4 waves on
// the same QR query rows; group g takes the key tiles g, g + 2, ... with its own LDS buffers, and the
// partial results (row statistics, output tile) meet in LDS at the end: the 2 waves a SIMD holds
// have the same amount of work from start to end.  With 128 rows each wave of a group has rows of its own
// and takes whole key tiles, with 64 two of them share 32 rows and take half of the keys of a tile each
// (which of the two: query_rows).
constexpr int kNT2 = 2 * kNT;
constexpr int kGroupLds = 4 * kTileB;                   // K and V tiles, two buffers each
constexpr int kXsOff = 2 * kGroupLds;                   // float [2 groups][2][128]: statistics exchange
constexpr size_t kQmSmem = 2 * kGroupLds + 2 * 2 * kBM * sizeof(float);

// What a wave takes with QR query rows per workgroup: query block qb and, of a group's four waves, part kp of the keys of
// every tile (KP parts); its partial results are number `part` of 2 KP.
template <int QR>
struct WaveShare {
    static constexpr int QB = QR / 32, KP = 4 / QB;
    int qb, kp, part;
    __device__ __forceinline__ WaveShare(int wid, int g) : qb(KP == 1 ? wid : wid % QB), kp(KP == 1 ? 0 : wid / QB), part(g * KP + kp) {}
};

// partial output tiles (DT x 16 floats per lane) 1 .. -> LDS -> added onto partial 0's; `region` ends at 2 kGroupLds
template <int QR, int DT>
__device__ __forceinline__ void merge_partials(float16_t (&acc)[DT], unsigned char *smem, const WaveShare<QR> &w, int tig)
{
    constexpr int NP = 2 * WaveShare<QR>::KP, NL = WaveShare<QR>::QB * 64, ONE = DT * 16 * NL;
    static_assert((NP - 1) * ONE * 4 <= 2 * kGroupLds - QR * kRowB, "beside the staged rows");
    float *x = reinterpret_cast<float *>(smem + 2 * kGroupLds - (NP - 1) * ONE * 4) + (tig & (NL - 1));
    if (w.part > 0) {
        float *mine = NP == 2 ? x : x + (w.part - 1) * ONE;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) mine[(dt * 16 + r) * NL] = acc[dt][r];
    }
    __syncthreads();
    if (w.part == 0) {
#pragma unroll
        for (int n = 0; n < NP - 1; n++)
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int r = 0; r < 16; r++) acc[dt][r] += x[n * ONE + (dt * 16 + r) * NL];
    }
}

// ---------------------------------------------------------------------------------------------
// Workgroups take the tiles in descending order of their key count; a CU holds one workgroup at a
// time (LDS), so the dispatcher hands the next tile to whichever CU is done first.
template <int KS, int DT, bool FAST, bool DMA, int QR>
__global__ void __launch_bounds__(kNT2, 2) attn_fwd_kernel(AttnArgs p)
{
    // the whole argument block in scalar registers at once (read field by field where the control flow first
    // wants it, it costs several dependent round trips to memory before the first tile is requested)
    asm volatile("" ::"s"(p.S), "s"(p.H), "s"(p.Dh), "s"(p.ld), "s"(p.alpha), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.dO),
                 "s"(p.o), "s"(p.out), "s"(p.dq), "s"(p.dk), "s"(p.dv), "s"(p.m), "s"(p.l), "s"(p.y), "s"(p.sig),
                 "s"(p.acc_dq), "s"(p.acc_dk), "s"(p.acc_dv));
    typedef AttnMath<FAST> M;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    if constexpr (!DMA) zero_lds(smem, 2 * kGroupLds);   // the pad columns of the tile buffers: zero from here on
    // wave-uniform values kept in scalar registers, so that the branches on them are scalar branches
    const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tig = threadIdx.x & (kNT - 1);
    unsigned char *Ks = smem + g * kGroupLds, *Vs = Ks + 2 * kTileB;
    float *xs = reinterpret_cast<float *>(smem + kXsOff);
    const int lane = tig & 63, wid = __builtin_amdgcn_readfirstlane(tig >> 6), l32 = lane & 31, lh = lane >> 5;
    const int S = p.S, Dh = p.Dh;
    const int64_t ld = p.ld;
    const int nqt = (S + QR - 1) / QR;
    const WaveShare<QR> ws(wid, g);
    constexpr int KP = WaveShare<QR>::KP, NP = 2 * KP;
    const int h = blockIdx.x % p.H, qt = nqt - 1 - blockIdx.x / p.H;
    const int shift = DMA ? (int)(((int64_t)h * Dh) & 7) : 0;          // the head's first column in its window
    gptr_t Q = gp(p.q) + (int64_t)h * Dh, K = gp(p.k) + (int64_t)h * Dh - shift, V = gp(p.v) + (int64_t)h * Dh - shift;
    {
        const int i0 = qt * QR, qrow = ws.qb * 32 + l32, r0 = i0 + ws.qb * 32, myrow = r0 + l32;

        // the queries: with direct tiles they come as two tiles straight into LDS below, beside the first key
        // and value tiles (a load in which every lane addresses its own row is served at one lane per clock)
        half8_t qf[KS];
        if constexpr (!DMA) load_frags<KS>(qf, Q, ld, myrow, S, Dh, lh, shift);

        const int kend = min(i0 + QR, S);                 // keys [0, kend) are visible to the tile
        const int njt = (kend + kTileRows - 1) / kTileRows, niter = (njt + 1) / 2;
        typedef typename std::conditional<DMA, DmaTileMap, FastTileMap>::type Map;
        typedef typename std::conditional<DMA, DmaTileLoader, FastTileLoader>::type Loader;
        const Map tm(ld, Dh, shift);
        Loader tk, tv;

        // ---- pass 1: row maximum and sum; each lane over its half of the keys of its group's tiles
        float m_run = -INFINITY, l_run = 0.f;
        if (g < njt) {
            tk.load(tm, K + (int64_t)g * kTileRows * ld, S - g * kTileRows, Ks);
            tk.store(tm, Ks);
            // the V buffers idle through pass 1: the first V tile of pass 2 comes in now
            if constexpr (DMA) tv.load(tm, V + (int64_t)g * kTileRows * ld, S - g * kTileRows, Vs);
        }
        if constexpr (DMA) {
            // rows 64 g .. 64 g + 63 of the workgroup's queries into this group's second V buffer, which idles
            // until the second pass; every wave then takes its fragments from the tile that holds its rows
            if (QR > 64 || g == 0)
                tv.load(tm, Q - shift + (int64_t)(i0 + g * kTileRows) * ld, S - (i0 + g * kTileRows), Vs + kTileB);
            zero_pads(smem, 2 * kGroupLds / kRowB, (Dh + shift + 7) >> 3);
        }
        tile_sync<DMA>();
        if constexpr (DMA)
            frags_from_tile<KS>(qf, smem + (ws.qb >> 1) * kGroupLds + 3 * kTileB, (ws.qb & 1) * 32 + l32, Dh, lh, shift);
        int it0 = 0;
        if constexpr (FAST && KP == 1) {
            // The key tiles wholly below the diagonal for every wave (iterations 0 .. qt - 1 of both groups) as a
            // pipeline: the products of a score tile run while the statistics of the tile before it are updated.
            // The same operations on the same values in the same order as the general loop below.
            // in 8 pieces: round the scores; their maximum; 4 x (4 exponentials and their sum); the running pair
            half2v_t sp[8];
            float m_new, cexp, sum;
            auto stat_piece = [&](const float16_t &acc, auto i_c) __attribute__((always_inline)) {
                constexpr int i = decltype(i_c)::value;
                if constexpr (i == 0) {
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        sp[e] = __builtin_convertvector(float2v_t{scaled(p.alpha, acc[2 * e]), scaled(p.alpha, acc[2 * e + 1])}, half2v_t);
                } else if constexpr (i == 1) {
                    half2v_t mx = sp[0];
#pragma unroll
                    for (int e = 1; e < 8; e++) mx = __builtin_elementwise_max(mx, sp[e]);
                    m_new = fmaxf(m_run, (float)__builtin_fmaxf16(mx[0], mx[1]));
                    cexp = m_new * kLog2e;
                    sum = 0.f;
                } else if constexpr (i < 6) {
#pragma unroll
                    for (int e = 4 * (i - 2); e < 4 * (i - 1); e++) sum += exp2_mix(sp[e >> 1][e & 1], cexp);
                } else if constexpr (i == 6) {
                    l_run = ((m_run == -INFINITY) ? 0.f : l_run * M::ex(m_run, m_new)) + sum;
                    m_run = m_new;
                }
            };
            auto stat_full = [&](const float16_t &acc) __attribute__((always_inline)) {
                stat_piece(acc, std::integral_constant<int, 0>{});
                stat_piece(acc, std::integral_constant<int, 1>{});
                stat_piece(acc, std::integral_constant<int, 2>{});
                stat_piece(acc, std::integral_constant<int, 3>{});
                stat_piece(acc, std::integral_constant<int, 4>{});
                stat_piece(acc, std::integral_constant<int, 5>{});
                stat_piece(acc, std::integral_constant<int, 6>{});
            };
            const int nfull = min(qt, niter);
            if (nfull > 0) {
                float16_t accp = prod_direct<KS>(Ks, 0, qf, l32, lh);
                for (int it = 0; it < nfull; it++) {
                    const int jt = 2 * it + g, cur = it & 1;
                    const bool nxt = jt + 2 < njt;
                    if (nxt) tk.load(tm, K + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Ks + (cur ^ 1) * kTileB);
                    accp = prod_direct_with<KS, 7>(Ks + cur * kTileB, 32, qf, l32, lh, [&](auto i_c) { stat_piece(accp, i_c); });
                    if (nxt) tk.store(tm, Ks + (cur ^ 1) * kTileB);
                    tile_sync<DMA>();
                    if (it + 1 < nfull)
                        accp = prod_direct_with<KS, 7>(Ks + (cur ^ 1) * kTileB, 0, qf, l32, lh, [&](auto i_c) { stat_piece(accp, i_c); });
                    else
                        stat_full(accp);
                }
                it0 = nfull;
            }
        }
        for (int it = it0; it < niter; it++) {
            const int jt = 2 * it + g, cur = it & 1;
            const bool nxt = jt + 2 < njt;
            if (nxt) tk.load(tm, K + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Ks + (cur ^ 1) * kTileB);
            if (jt < njt) {
#pragma unroll
                for (int k2 = 0; k2 < 2 / KP; k2++) {
                    const int kt = KP == 1 ? k2 : ws.kp, kb = jt * kTileRows + 32 * kt;
                    if (kb > r0 + 31) continue;          // every key of the tile is beyond every row of the wave
                    const float16_t acc = prod_direct<KS>(Ks + cur * kTileB, 32 * kt, qf, l32, lh);
                    const bool full = kb + 31 <= r0;
                    float sv[16], mt = -INFINITY, sum = 0.f;
                    if constexpr (FAST) {
                        half_t sh[16];
                        if (full) {
#pragma unroll
                            for (int e = 0; e < 16; e++) sh[e] = f2h(scaled(p.alpha, acc[e]));
                        } else {
#pragma unroll
                            for (int e = 0; e < 16; e++) {
                                const int key = kb + 8 * (e >> 2) + 4 * lh + (e & 3);
                                sh[e] = key <= myrow ? f2h(scaled(p.alpha, acc[e])) : (half_t)-INFINITY;
                            }
                        }
                        const float m_new = fmaxf(m_run, max16(sh)), c = m_new * kLog2e;
                        if (full) {
#pragma unroll
                            for (int e = 0; e < 16; e++) sum += exp2_mix(sh[e], c);
                        } else {
#pragma unroll
                            for (int e = 0; e < 16; e++)
                                sum += (sh[e] == (half_t)-INFINITY) ? 0.f : exp2_mix(sh[e], c);
                        }
                        l_run = ((m_run == -INFINITY) ? 0.f : l_run * M::ex(m_run, m_new)) + sum;
                        m_run = m_new;
                    } else if (full) {                   // no masks on tiles wholly below the diagonal
#pragma unroll
                        for (int e = 0; e < 16; e++) {
                            sv[e] = rnd16(scaled(p.alpha, acc[e]));
                            mt = fmaxf(mt, sv[e]);
                        }
                        const float m_new = fmaxf(m_run, mt);
#pragma unroll
                        for (int e = 0; e < 16; e++) sum += M::ex(sv[e], m_new);
                        l_run = ((m_run == -INFINITY) ? 0.f : l_run * M::ex(m_run, m_new)) + sum;
                        m_run = m_new;
                    } else {
#pragma unroll
                        for (int e = 0; e < 16; e++) {
                            const int key = kb + 8 * (e >> 2) + 4 * lh + (e & 3);
                            const float s = rnd16(scaled(p.alpha, acc[e]));
                            sv[e] = key <= myrow ? s : -INFINITY;
                            mt = fmaxf(mt, sv[e]);
                        }
                        const float m_new = fmaxf(m_run, mt);
#pragma unroll
                        for (int e = 0; e < 16; e++) sum += (sv[e] == -INFINITY) ? 0.f : M::ex(sv[e], m_new);
                        l_run = ((m_run == -INFINITY) ? 0.f : l_run * M::ex(m_run, m_new)) + sum;
                        m_run = m_new;
                    }
                }
            }
            if (nxt) tk.store(tm, Ks + (cur ^ 1) * kTileB);
            tile_sync<DMA>();
        }
        // pass 2 starts from the group's first K tile again: on its way while the statistics are merged
        if constexpr (DMA) {
            if (g < njt) tk.load(tm, K + (int64_t)g * kTileRows * ld, S - g * kTileRows, Ks);
        }
        float m, l;
        {
            // the partial (maximum, sum) pairs of a row -- two lanes in each wave that holds it -- merged
            // in one fixed order by every lane that needs the result
            const float m_o = __shfl_xor(m_run, 32, 64), l_o = __shfl_xor(l_run, 32, 64);
            const float ma = lh ? m_o : m_run, la = lh ? l_o : l_run;
            const float mb = lh ? m_run : m_o, lb = lh ? l_run : l_o;
            const float mg = fmaxf(ma, mb);
            const float lg = ((ma == -INFINITY) ? 0.f : la * M::ex(ma, mg)) + ((mb == -INFINITY) ? 0.f : lb * M::ex(mb, mg));
            if (lh == 0) {
                xs[(ws.part * 2 + 0) * QR + qrow] = mg;
                xs[(ws.part * 2 + 1) * QR + qrow] = lg;
            }
            __syncthreads();
            m = xs[qrow];
#pragma unroll
            for (int n = 1; n < NP; n++) m = fmaxf(m, xs[2 * n * QR + qrow]);
            l = 0.f;
#pragma unroll
            for (int n = 0; n < NP; n++) {
                const float mn = xs[2 * n * QR + qrow], ln = xs[(2 * n + 1) * QR + qrow];
                const float e = (mn == -INFINITY) ? 0.f : ln * M::ex(mn, m);
                l = n ? l + e : e;
            }
            if (myrow >= S) { m = 0.f; l = 1.f; }
            if (ws.part == 0 && lh == 0 && myrow < S) {
                p.m[(int64_t)h * S + myrow] = m;
                p.l[(int64_t)h * S + myrow] = l;
            }
        }
        const float y = recip_refined(l);
        const float cs = prob_shift(m, l);

        // ---- pass 2: probabilities and O
        float16_t oacc[DT];
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) oacc[dt][r] = 0.f;
        if (!DMA && g < njt) {
            tk.load(tm, K + (int64_t)g * kTileRows * ld, S - g * kTileRows, Ks);
            tv.load(tm, V + (int64_t)g * kTileRows * ld, S - g * kTileRows, Vs);
            tk.store(tm, Ks);
            tv.store(tm, Vs);
        }
        tile_sync<DMA>();
        int it2 = 0;
        if constexpr (FAST && DMA && KP == 1) {
            // The key tiles wholly below the diagonal for every wave, as in pass 1, with the vector arithmetic of a
            // block between the MFMAs of its neighbours: per tile, the scores of its second block are formed while
            // the probabilities of the first are, the first block's P V products run while the second's
            // probabilities are formed, then the second's P V; the first scores of the next tile follow the barrier
            // that publishes it (the P V products read the V tile, which the next iteration's loads overwrite, so
            // they cannot move behind the barrier).  The same operations on the same values in the same order as the
            // general loop below.
            const int nfull = min(qt, niter);
            if (nfull > 0) {
                half2v_t sp[8];
                float pe[16];
                half8_t pk[2][2];                               // packed probabilities of the tile's two blocks
                auto prob_piece = [&](const float16_t &acc, half8_t (&out)[2], auto i_c) __attribute__((always_inline)) {
                    constexpr int i = decltype(i_c)::value;
                    if constexpr (i == 0) {
#pragma unroll
                        for (int e = 0; e < 8; e++)
                            sp[e] = __builtin_convertvector(float2v_t{scaled(p.alpha, acc[2 * e]), scaled(p.alpha, acc[2 * e + 1])}, half2v_t);
                    } else if constexpr (i < 5) {
#pragma unroll
                        for (int e = 4 * (i - 1); e < 4 * i; e++) pe[e] = exp2_mix(sp[e >> 1][e & 1], cs);
                    } else {
                        out[0] = pack8(pe);
                        out[1] = pack8(pe + 8);
                    }
                };
                float16_t accp = prod_direct<KS>(Ks, 0, qf, l32, lh);
                for (int it = 0; it < nfull; it++) {
                    const int jt = 2 * it + g, cur = it & 1;
                    const bool nxt = jt + 2 < njt;
                    if (nxt) {
                        tk.load(tm, K + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Ks + (cur ^ 1) * kTileB);
                        tv.load(tm, V + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Vs + (cur ^ 1) * kTileB);
                    }
                    const float16_t acc2 = prod_direct_with<KS, 6>(Ks + cur * kTileB, 32, qf, l32, lh,
                                                                   [&](auto i_c) { prob_piece(accp, pk[0], i_c); });
                    asm volatile("" : "+v"(pk[0][0]), "+v"(pk[0][1]));
                    prod_tr_with<DT, 6>(oacc, Vs + cur * kTileB, 0, pk[0][0], pk[0][1], lane,
                                        [&](auto i_c) { prob_piece(acc2, pk[1], i_c); });
                    asm volatile("" : "+v"(pk[1][0]), "+v"(pk[1][1]));
                    prod_tr<DT>(oacc, Vs + cur * kTileB, 32, pk[1][0], pk[1][1], lane);
                    tile_sync<DMA>();
                    if (it + 1 < nfull) accp = prod_direct<KS>(Ks + (cur ^ 1) * kTileB, 0, qf, l32, lh);
                }
                it2 = nfull;
            }
        }
        for (int it = it2; it < niter; it++) {
            const int jt = 2 * it + g, cur = it & 1;
            const bool nxt = jt + 2 < njt;
            if (nxt) {
                tk.load(tm, K + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Ks + (cur ^ 1) * kTileB);
                tv.load(tm, V + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Vs + (cur ^ 1) * kTileB);
            }
            if (jt < njt) {
#pragma unroll
                for (int k2 = 0; k2 < 2 / KP; k2++) {
                    const int kt = KP == 1 ? k2 : ws.kp, kb = jt * kTileRows + 32 * kt;
                    if (kb > r0 + 31) continue;
                    const float16_t acc = prod_direct<KS>(Ks + cur * kTileB, 32 * kt, qf, l32, lh);
                    const bool full = kb + 31 <= r0;
                    float pe[16];
                    if constexpr (FAST) {
                        if (full) {
#pragma unroll
                            for (int e = 0; e < 16; e++) pe[e] = exp2_mix(f2h(scaled(p.alpha, acc[e])), cs);
                        } else {
#pragma unroll
                            for (int e = 0; e < 16; e++) {
                                const int key = kb + 8 * (e >> 2) + 4 * lh + (e & 3);
                                pe[e] = key <= myrow ? exp2_mix(f2h(scaled(p.alpha, acc[e])), cs) : 0.f;
                            }
                        }
                    } else if (full) {
#pragma unroll
                        for (int e = 0; e < 16; e++) pe[e] = M::prob(rnd16(scaled(p.alpha, acc[e])), m, l, y);
                    } else {
#pragma unroll
                        for (int e = 0; e < 16; e++) {
                            const int key = kb + 8 * (e >> 2) + 4 * lh + (e & 3);
                            const float pr_ = M::prob(rnd16(scaled(p.alpha, acc[e])), m, l, y);
                            pe[e] = key <= myrow ? pr_ : 0.f;
                        }
                    }
                    prod_tr<DT>(oacc, Vs + cur * kTileB, 32 * kt, pack8(pe), pack8(pe + 8), lane);
                }
            }
            if (nxt) {
                tk.store(tm, Ks + (cur ^ 1) * kTileB);
                tv.store(tm, Vs + (cur ^ 1) * kTileB);
            }
            tile_sync<DMA>();
        }
        merge_partials<QR, DT>(oacc, smem, ws, tig);
        if constexpr (DMA) {
            if (ws.part == 0) stage_rows<DT>(smem, oacc, qrow, lh, 1.0f);
            __syncthreads();
            write_rows(smem, p.out + (int64_t)i0 * ld + (int64_t)h * Dh - shift, ld, min(QR, S - i0), Dh, shift,
                       threadIdx.x, kNT2);
        } else if (ws.part == 0 && myrow < S) {
            half_t *orow = p.out + (int64_t)myrow * ld + (int64_t)h * Dh;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int d0 = 32 * dt + 8 * q + 4 * lh - shift;
                    if (d0 >= 0 && d0 < Dh)
                        store_row4(orow + d0, oacc[dt][4 * q], oacc[dt][4 * q + 1], oacc[dt][4 * q + 2],
                                   oacc[dt][4 * q + 3], 1.0f, 0);
                }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// dQ: queries fixed, loop over the key tiles at or before them, work split as in the forward kernel.
// Pass 0 forms sigma = sum_j P' f32(dP16); pass 1 dS16 and dQ.  Leaves y = 1 / l and sigma per row for
// the dK / dV kernel.
template <int KS, int DT, bool FAST, bool DMA, int QR>
__global__ void __launch_bounds__(kNT2, 2) attn_bwd_dq_kernel(AttnArgs p)
{
    // the whole argument block in scalar registers at once (read field by field where the control flow first
    // wants it, it costs several dependent round trips to memory before the first tile is requested)
    asm volatile("" ::"s"(p.S), "s"(p.H), "s"(p.Dh), "s"(p.ld), "s"(p.alpha), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.dO),
                 "s"(p.o), "s"(p.out), "s"(p.dq), "s"(p.dk), "s"(p.dv), "s"(p.m), "s"(p.l), "s"(p.y), "s"(p.sig),
                 "s"(p.acc_dq), "s"(p.acc_dk), "s"(p.acc_dv));
    typedef AttnMath<FAST> M;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tig = threadIdx.x & (kNT - 1);
    unsigned char *Ks = smem + g * kGroupLds, *Vs = Ks + 2 * kTileB;
    float *xs = reinterpret_cast<float *>(smem + kXsOff);
    const int lane = tig & 63, wid = __builtin_amdgcn_readfirstlane(tig >> 6), l32 = lane & 31, lh = lane >> 5;
    const int S = p.S, Dh = p.Dh;
    const int64_t ld = p.ld;
    const int nqt = (S + QR - 1) / QR;
    const WaveShare<QR> ws(wid, g);
    constexpr int KP = WaveShare<QR>::KP, NP = 2 * KP;
    const int h = blockIdx.x % p.H, qt = nqt - 1 - blockIdx.x / p.H;
    const int64_t hoff = (int64_t)h * Dh;
    const int shift = DMA ? (int)(hoff & 7) : 0;                        // the head's first column in its window
    // the pad columns of the tile buffers: zero from the first barrier on (direct tiles: cleared below, behind
    // the first loads)
    if constexpr (!DMA) zero_lds(smem, 2 * kGroupLds);
    gptr_t K = gp(p.k) + hoff - shift, V = gp(p.v) + hoff - shift;
    {
        const int i0 = qt * QR, qrow = ws.qb * 32 + l32, r0 = i0 + ws.qb * 32, myrow = r0 + l32;
        const int kend = min(i0 + QR, S);
        const int njt = (kend + kTileRows - 1) / kTileRows, niter = (njt + 1) / 2;
        typedef typename std::conditional<DMA, DmaTileMap, TileMap8>::type Map;
        typedef typename std::conditional<DMA, DmaTileLoader, TileLoader8>::type Loader;
        const Map tm(ld, Dh, shift);
        Loader tk, tv;
        auto first_tiles = [&]() __attribute__((always_inline)) {
            if (g < njt) {
                tk.load(tm, K + (int64_t)g * kTileRows * ld, S - g * kTileRows, Ks);
                tv.load(tm, V + (int64_t)g * kTileRows * ld, S - g * kTileRows, Vs);
                tk.store(tm, Ks);
                tv.store(tm, Vs);
            }
        };
        // The fixed operands.  A load in which every lane addresses its own row is served at about one lane
        // per clock and CU (42 such instructions in each of 8 waves: 21 k of the 29 k cycles this kernel used
        // to spend before its first product), so with direct tiles the workgroup's 128 rows of q, dO and the
        // forward output (used by the short form of sigma, decided below from the statistics) come as six
        // tiles straight into LDS, whole row segments per instruction, and each wave picks its fragments out
        // of them; both wave groups hold the same rows and share the tiles.  Then the first key and value
        // tiles go out, into the same buffers, before anything else is computed.
        bool tiles_on_the_way = false;
        float m = ((gfptr_t)p.m)[(int64_t)h * S + min(myrow, S - 1)];
        float l = ((gfptr_t)p.l)[(int64_t)h * S + min(myrow, S - 1)];
        // the row this lane votes for on the form of sigma below: of the 128 rows the workgroup's are part of
        const int vrow = QR == 128 ? myrow : (i0 & ~127) + (threadIdx.x & 127);
        const float lvote = QR == 128 ? l : ((gfptr_t)p.l)[(int64_t)h * S + min(vrow, S - 1)];
        half8_t qf[KS], gf[KS], of[FAST ? KS : 1];
        if constexpr (DMA) {
            const int first = i0 + (QR > 64 ? g * kTileRows : 0), left = S - first;
            const int64_t off = hoff - shift + (int64_t)first * ld;
            const bool want_o = FAST && p.o;
            if (QR > 64) {
                tk.load(tm, gp(p.q) + off, left, smem + g * kTileB);
                tk.load(tm, gp(p.dO) + off, left, smem + (2 + g) * kTileB);
                if (want_o) tk.load(tm, gp(p.o) + off, left, smem + (4 + g) * kTileB);
            } else {                              // three tiles, two groups
                tk.load(tm, (g ? gp(p.dO) : gp(p.q)) + off, left, smem + 2 * g * kTileB);
                if (want_o && g) tk.load(tm, gp(p.o) + off, left, smem + 4 * kTileB);
            }
            zero_pads(smem, 2 * kGroupLds / kRowB, (Dh + shift + 7) >> 3);
            tile_sync<DMA>();
            const unsigned char *mine = smem + (ws.qb >> 1) * kTileB;
            const int trow = (ws.qb & 1) * 32 + l32;
            frags_from_tile<KS>(qf, mine, trow, Dh, lh, shift);
            frags_from_tile<KS>(gf, mine + 2 * kTileB, trow, Dh, lh, shift);
            if constexpr (FAST) {
                if (want_o) frags_from_tile<KS>(of, mine + 4 * kTileB, trow, Dh, lh, shift);
            }
            __syncthreads();                      // every wave holds its fragments: the buffers are free again
            first_tiles();
            tiles_on_the_way = true;
        } else {
            load_frags<KS>(qf, gp(p.q) + hoff, ld, myrow, S, Dh, lh, shift);
            load_frags<KS>(gf, gp(p.dO) + hoff, ld, myrow, S, Dh, lh, shift);
            if constexpr (FAST) {
                if (p.o) load_frags<KS>(of, gp(p.o) + hoff, ld, myrow, S, Dh, lh, shift);
            }
        }
        float sig = 0.f;
        if (myrow >= S) {
            m = 0.f;
            l = 1.f;
        }
        const float y = recip_refined(l);
        const float cs = prob_shift(m, l);

        float16_t dacc[DT];
        auto run_pass = [&](auto pass_c) __attribute__((always_inline)) {
            constexpr int PASS = decltype(pass_c)::value;
            float part = 0.f;
            if (!tiles_on_the_way) first_tiles();
            tiles_on_the_way = false;
            tile_sync<DMA>();
            int it0 = 0;
            if constexpr (FAST && DMA && KP == 1 && PASS == 1 && KS == 4) {
                // The key tiles wholly below the diagonal for every wave, as in the forward kernel, with the vector arithmetic
                // between MFMAs: that of a tile's first block between the score and dP products of its second, the second's
                // between the first's products with K; the first block's scores and dP of the next tile follow the barrier
                // that publishes it.  The same operations on the same values in the same order as the general loop below.
                // Heads to 64: 1531 positions, 32 heads 54.4 -> 44.9 us, 1000, 40 heads 37.0 -> 30.4, 4000, 16 heads 92 -> 80.
                // Wider ones have no registers for it: 32 heads of 100 at 2048 positions spill 23 and take 102 us instead of
                // 91; with fragments read three ahead instead of all there is no spill in the loop, and 99.
                const int nfull = min(qt, niter);
                if (nfull > 0) {
                    half2v_t sp[8], dp[8];
                    float pr[16], de[16];
                    half8_t pk[2][2];                           // packed dS of the tile's two blocks
                    auto prob_piece = [&](const float16_t &sacc, const float16_t &pacc, auto i_c) __attribute__((always_inline)) {
                        constexpr int i = decltype(i_c)::value;
                        if constexpr (i == 1) {
#pragma unroll
                            for (int e = 0; e < 8; e++)
                                sp[e] = __builtin_convertvector(float2v_t{scaled(p.alpha, sacc[2 * e]), scaled(p.alpha, sacc[2 * e + 1])}, half2v_t);
                        } else if constexpr (i > 1) {
#pragma unroll
                            for (int e = 4 * (i - 2); e < 4 * (i - 1); e++) pr[e] = exp2_mix(sp[e >> 1][e & 1], cs);
                        } else {
#pragma unroll
                            for (int e = 0; e < 8; e++) dp[e] = __builtin_convertvector(float2v_t{pacc[2 * e], pacc[2 * e + 1]}, half2v_t);
                        }
                    };
                    auto ds_piece = [&](half8_t (&out)[2], auto i_c) __attribute__((always_inline)) {
                        constexpr int i = decltype(i_c)::value;
                        if constexpr (i < 4) {
#pragma unroll
                            for (int e = 4 * i; e < 4 * i + 4; e++) de[e] = __builtin_fmaf((float)dp[e >> 1][e & 1], pr[e], -(sig * pr[e]));
                        } else {
                            out[i - 4] = pack8(de + 8 * (i - 4));
                        }
                    };
                    float16_t s0 = prod_direct<KS>(Ks, 0, qf, l32, lh), p0 = prod_direct<KS>(Vs, 0, gf, l32, lh);
                    for (int it = 0; it < nfull; it++) {
                        const int jt = 2 * it + g, cur = it & 1;
                        const unsigned char *Kc = Ks + cur * kTileB, *Vc = Vs + cur * kTileB;
                        if (jt + 2 < njt) {
                            tk.load(tm, K + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Ks + (cur ^ 1) * kTileB);
                            tv.load(tm, V + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Vs + (cur ^ 1) * kTileB);
                        }
                        const float16_t s1 = prod_direct_with<KS, 6>(Kc, 32, qf, l32, lh, [&](auto i_c) { prob_piece(s0, p0, i_c); });
                        const float16_t p1 = prod_direct_with<KS, 6>(Vc, 32, gf, l32, lh, [&](auto i_c) { ds_piece(pk[0], i_c); });
                        asm volatile("" : "+v"(pk[0][0]), "+v"(pk[0][1]));
                        prod_tr_with<DT, 8>(dacc, Kc, 0, pk[0][0], pk[0][1], lane, [&](auto i_c) __attribute__((always_inline)) {
                            constexpr int i = decltype(i_c)::value;
                            if constexpr (i < 6) {
                                prob_piece(s1, p1, i_c);
                            } else {
                                ds_piece(pk[1], std::integral_constant<int, 2 * (i - 6)>{});
                                ds_piece(pk[1], std::integral_constant<int, 2 * (i - 6) + 1>{});
                                ds_piece(pk[1], std::integral_constant<int, i - 2>{});
                            }
                        });
                        asm volatile("" : "+v"(pk[1][0]), "+v"(pk[1][1]));
                        prod_tr<DT>(dacc, Kc, 32, pk[1][0], pk[1][1], lane);
                        tile_sync<DMA>();
                        if (it + 1 < nfull) {
                            s0 = prod_direct<KS>(Ks + (cur ^ 1) * kTileB, 0, qf, l32, lh);
                            p0 = prod_direct<KS>(Vs + (cur ^ 1) * kTileB, 0, gf, l32, lh);
                        }
                    }
                    it0 = nfull;
                }
            }
            for (int it = it0; it < niter; it++) {
                const int jt = 2 * it + g, cur = it & 1;
                const bool nxt = jt + 2 < njt;
                if (nxt) {
                    tk.load(tm, K + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Ks + (cur ^ 1) * kTileB);
                    tv.load(tm, V + (int64_t)(jt + 2) * kTileRows * ld, S - (jt + 2) * kTileRows, Vs + (cur ^ 1) * kTileB);
                }
                // 32 keys of the tile
                auto block = [&](int kt) __attribute__((always_inline)) {
                    const int kb = jt * kTileRows + 32 * kt;
                    if (kb > r0 + 31) return;
                    const float16_t sacc = prod_direct<KS>(Ks + cur * kTileB, 32 * kt, qf, l32, lh);
                    const float16_t pacc = prod_direct<KS>(Vs + cur * kTileB, 32 * kt, gf, l32, lh);
                    const bool full = kb + 31 <= r0;
                    float de[16];
                    if constexpr (FAST) {
                        // sigma and dS with the f16 value of dP read by the fused multiply-add
                        half_t dph[16];
                        round16(dph, pacc);
                        if (full) {
#pragma unroll
                            for (int e = 0; e < 16; e++) {
                                const float pr_ = exp2_mix(f2h(scaled(p.alpha, sacc[e])), cs);
                                const half_t dp = dph[e];
                                if (PASS == 0) part = __builtin_fmaf((float)dp, pr_, part);
                                else de[e] = __builtin_fmaf((float)dp, pr_, -(sig * pr_));
                            }
                        } else {
#pragma unroll
                            for (int e = 0; e < 16; e++) {
                                const bool live = kb + 8 * (e >> 2) + 4 * lh + (e & 3) <= myrow;
                                const float pr_ = exp2_mix(f2h(scaled(p.alpha, sacc[e])), cs);
                                const half_t dp = dph[e];
                                if (PASS == 0) part += live ? (float)dp * pr_ : 0.f;
                                else de[e] = live ? __builtin_fmaf((float)dp, pr_, -(sig * pr_)) : 0.f;
                            }
                        }
                    } else if (full) {
#pragma unroll
                        for (int e = 0; e < 16; e++) {
                            const float pr_ = M::prob(rnd16(scaled(p.alpha, sacc[e])), m, l, y);
                            const float tt = pr_ * rnd16(pacc[e]);
                            if (PASS == 0) part += tt;
                            else de[e] = tt - sig * pr_;
                        }
                    } else {
#pragma unroll
                        for (int e = 0; e < 16; e++) {
                            const bool live = kb + 8 * (e >> 2) + 4 * lh + (e & 3) <= myrow;
                            const float pr_ = M::prob(rnd16(scaled(p.alpha, sacc[e])), m, l, y);
                            const float tt = pr_ * rnd16(pacc[e]);
                            if (PASS == 0) part += live ? tt : 0.f;
                            else de[e] = live ? tt - sig * pr_ : 0.f;
                        }
                    }
                    if (PASS == 1) prod_tr<DT>(dacc, Ks + cur * kTileB, 32 * kt, pack8(de), pack8(de + 8), lane);
                };
                if (jt < njt) {
                    if constexpr (KP == 2) {
                        block(ws.kp);
                    } else if constexpr (PASS == 0) {
                        // one piece of code for both: only the first workgroup of a head runs this pass, and meets every
                        // instruction of it once
#pragma unroll 1
                        for (int kt = 0; kt < 2; kt++) block(kt);
                    } else {
#pragma unroll
                        for (int kt = 0; kt < 2; kt++) block(kt);
                    }
                }
                if (nxt) {
                    tk.store(tm, Ks + (cur ^ 1) * kTileB);
                    tv.store(tm, Vs + (cur ^ 1) * kTileB);
                }
                tile_sync<DMA>();
            }
            return part;
        };
        // sigma_i = sum_j P'_ij f32(dP16_ij).  In exact arithmetic that is sum_d dO_id O_id, which needs no pass
        // over the keys; in the reference's arithmetic the two differ by the f16 roundings of dP16, P16 and O,
        // about 2^-11 |dP| sqrt(sum_j P_ij^2).  Where a row's probability mass is spread that is below the
        // rounding of dS16 itself.  Where it sits on one key it is not: the reference has dP16 - sigma = 0
        // there exactly, and rows 0 and 1 of a sequence failed the element bound with the short form.  So
        // 128 rows (of one workgroup or two) take the short form only if every one of them has sum_j
        // exp(S16_ij - m_i) >= kSpread (no probability above 1 / kSpread), else the pass over the keys; the
        // exactly rounded build always takes the pass.
        bool short_sigma = false;
        if constexpr (FAST) {
            if (p.o) short_sigma = __syncthreads_and(vrow >= S || lvote >= kSpread) != 0;
        }
        if (short_sigma) {
            float part = 0.f;
#pragma unroll
            for (int ks = 0; ks < (FAST ? KS : 1); ks++)
#pragma unroll
                for (int e = 0; e < 8; e++) part = __builtin_fmaf((float)gf[ks][e], (float)of[ks][e], part);
            sig = with32(part, OpSum());                     // the two lanes of a row
        } else {
            const float part = run_pass(std::integral_constant<int, 0>{});
            const float pg = with32(part, OpSum());         // the two lanes of a row, then the waves that hold it
            if (lh == 0) xs[ws.part * QR + qrow] = pg;
            __syncthreads();
            sig = xs[qrow];
#pragma unroll
            for (int n = 1; n < NP; n++) sig += xs[n * QR + qrow];
        }
        if (ws.part == 0 && lh == 0 && myrow < S) {
            p.y[(int64_t)h * S + myrow] = FAST ? cs : y;          // what the dK / dV kernel wants per row
            p.sig[(int64_t)h * S + myrow] = sig;
        }
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) dacc[dt][r] = 0.f;
        run_pass(std::integral_constant<int, 1>{});
        merge_partials<QR, DT>(dacc, smem, ws, tig);
        if (DMA && !p.acc_dq) {
            if (ws.part == 0) stage_rows<DT>(smem, dacc, qrow, lh, p.alpha);
            __syncthreads();
            write_rows(smem, p.dq + (int64_t)i0 * ld + hoff - shift, ld, min(QR, S - i0), Dh, shift, threadIdx.x, kNT2);
        } else if (ws.part == 0 && myrow < S) {
            half_t *drow = p.dq + (int64_t)myrow * ld + hoff;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int d0 = 32 * dt + 8 * q + 4 * lh - shift;
                    if (d0 >= 0 && d0 < Dh)
                        store_row4(drow + d0, dacc[dt][4 * q], dacc[dt][4 * q + 1], dacc[dt][4 * q + 2],
                                   dacc[dt][4 * q + 3], p.alpha, p.acc_dq);
                }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// dK, dV: keys fixed (128 or 64 per workgroup of 4 waves, a lane owns one), loop over the query tiles at or
// after them; the key tiles with the most queries first.

// tile buffers per tensor (Q, dO) and sets of row statistics
constexpr int dkv_bufs(int keys) { return keys == 128 ? 3 : 2; }

// SPLIT: a workgroup takes p.per of the query tiles of its keys and leaves its sums in p.part (dkv_parts).
// KR: keys per workgroup.  With 64 two waves share 32 keys and take one 32-query block of every tile each.
template <int KS, int DT, bool FAST, bool DMA, bool SPLIT, int KR>
__global__ void __launch_bounds__(kNT, KR == 64 && KS == 4 ? 2 : 1) attn_bwd_dkv_kernel(AttnArgs p)
{
    // the whole argument block in scalar registers at once (read field by field where the control flow first
    // wants it, it costs several dependent round trips to memory before the first tile is requested)
    asm volatile("" ::"s"(p.S), "s"(p.H), "s"(p.Dh), "s"(p.ld), "s"(p.alpha), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.dO),
                 "s"(p.o), "s"(p.out), "s"(p.dq), "s"(p.dk), "s"(p.dv), "s"(p.m), "s"(p.l), "s"(p.y), "s"(p.sig),
                 "s"(p.acc_dq), "s"(p.acc_dk), "s"(p.acc_dv));
    typedef AttnMath<FAST> M;
    constexpr int BUFS = dkv_bufs(KR);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *Qs = smem, *Gs = smem + BUFS * kTileB;
    float *St = reinterpret_cast<float *>(smem + 2 * BUFS * kTileB);   // [3][4][64]: m, l, y, sigma of a tile's rows
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31,
              lh = lane >> 5;
    const int S = p.S, Dh = p.Dh;
    const int64_t ld = p.ld;
    const int h = blockIdx.x % p.H, pz = blockIdx.x / p.H, pr = SPLIT ? pz / p.split : pz, z = SPLIT ? pz - pr * p.split : 0;
    static_assert(KR == 128 || (KR == 64 && DMA && !SPLIT), "keys of a workgroup");
    const int kb = KR == 128 ? wid : wid & 1, qh = KR == 128 ? 0 : wid >> 1;
    const int first_tile = pr * (KR / kTileRows) + z * (SPLIT ? p.per : 0);
    if (SPLIT && first_tile * kTileRows >= S) return;                   // no query tile left for this part
    const int64_t hoff = (int64_t)h * Dh;
    const int shift = DMA ? (int)(hoff & 7) : 0;                        // the head's first column in its window
    gptr_t Q = gp(p.q) + hoff - shift, G = gp(p.dO) + hoff - shift;
    // the pad columns of the tile buffers: zero from the first tile's barrier on (direct tiles: cleared below,
    // behind the first loads)
    if constexpr (!DMA) zero_lds(smem, 2 * BUFS * kTileB);
    // the four per-row statistics of a 64-query tile: lane t of wave w fetches array w, row t
    gfptr_t stat_src = (gfptr_t)(wid == 0 ? p.m : wid == 1 ? p.l : wid == 2 ? p.y : p.sig) + (int64_t)h * S;
    const float stat_pad = (wid == 1 || wid == 2) ? 1.f : 0.f;

    {
        const int kt_ = pr;                                             // low key tiles see the most queries
        const int c00 = kt_ * KR, c0 = c00 + kb * 32, mykey = c0 + l32;

        // the keys and values of the workgroup: with direct tiles they come as tiles straight into LDS, beside the
        // first query tile (below)
        half8_t kf[KS], vf[KS];
        if constexpr (!DMA) {
            load_frags<KS>(kf, gp(p.k) + hoff, ld, mykey, S, Dh, lh, shift);
            load_frags<KS>(vf, gp(p.v) + hoff, ld, mykey, S, Dh, lh, shift);
        }

        float16_t kacc[DT], vacc[DT];
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                kacc[dt][r] = 0.f;
                vacc[dt][r] = 0.f;
            }
        const int iq0 = first_tile, ntiles = (S + kTileRows - 1) / kTileRows, niq = SPLIT ? min(ntiles, iq0 + p.per) : ntiles;
        typedef typename std::conditional<DMA, DmaTileMap, FastTileMap>::type Map;
        typedef typename std::conditional<DMA, DmaTileLoader, FastTileLoader>::type Loader;
        const Map tm(ld, Dh, shift);
        Loader tq, tg;
        float st;
        auto load_stat = [&](int iq) __attribute__((always_inline)) {
            const int row = iq * kTileRows + lane;
            const float t = stat_src[row < S ? row : S - 1];
            st = row < S ? t : stat_pad;          // rows beyond S are masked; the pad only has to be finite
        };
        auto buf_of = [&](int iq) __attribute__((always_inline)) { return (iq - iq0) % BUFS; };
        auto fetch = [&](int iq) __attribute__((always_inline)) {        // tile iq on its way (registers or LDS)
            const int bf = buf_of(iq);
            tq.load(tm, Q + (int64_t)iq * kTileRows * ld, S - iq * kTileRows, Qs + bf * kTileB);
            tg.load(tm, G + (int64_t)iq * kTileRows * ld, S - iq * kTileRows, Gs + bf * kTileB);
            if constexpr (DMA) {
                // the statistics the same way (rows beyond S: the last row's, finite like the pad), so that no
                // register load stands between these loads and the point where the kernel waits for them
                const int row = min(iq * kTileRows + lane, S - 1);
                const uint32_t m0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(St + bf * 256 + wid * 64));
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                             :
                             : "s"(m0), "v"((uint32_t)row * 4u), "s"(stat_src)
                             : "memory");
            } else {
                load_stat(iq);
            }
        };
        auto land = [&](int iq) __attribute__((always_inline)) {         // ... into LDS, with its statistics
            const int bf = buf_of(iq);
            tq.store(tm, Qs + bf * kTileB);
            tg.store(tm, Gs + bf * kTileB);
            if constexpr (!DMA) St[bf * 256 + wid * 64 + lane] = st;
        };
        // one 32-query block of a tile, its three stages one after the other
        auto block = [&](int iq, int qb) __attribute__((always_inline)) {
            const int bf = buf_of(iq);
            const float *stc = St + bf * 256;
            const int qb0 = iq * kTileRows + 32 * qb;
            if (qb0 + 31 < c0 || qb0 >= S) return;        // every query of the block is before every key of the wave
            const float16_t sacc = prod_direct<KS, false>(Qs + bf * kTileB, 32 * qb, kf, l32, lh);
            const float16_t pacc = prod_direct<KS, false>(Gs + bf * kTileB, 32 * qb, vf, l32, lh);
            const bool full = qb0 >= c0 + 31 && qb0 + 32 <= S;
            float pe[16], de[16];
            half_t dph[16];
            if constexpr (FAST) round16(dph, pacc);
            auto elems = [&](auto full_c) __attribute__((always_inline)) {
                constexpr bool FULL = decltype(full_c)::value;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int qi = 32 * qb + 8 * q + 4 * lh;
                    float4_t mm, ll;
                    if constexpr (!FAST) {
                        mm = *reinterpret_cast<const float4_t *>(stc + 0 * 64 + qi);
                        ll = *reinterpret_cast<const float4_t *>(stc + 1 * 64 + qi);
                    }
                    const float4_t yy = *reinterpret_cast<const float4_t *>(stc + 2 * 64 + qi);
                    const float4_t sg = *reinterpret_cast<const float4_t *>(stc + 3 * 64 + qi);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int e = 4 * q + r, query = iq * kTileRows + qi + r;
                        float pr_, ds;
                        if constexpr (FAST) {                 // yy holds the exponent offset of the row
                            pr_ = exp2_mix(f2h(scaled(p.alpha, sacc[e])), yy[r]);
                            ds = __builtin_fmaf((float)dph[e], pr_, -(sg[r] * pr_));
                        } else {
                            pr_ = M::prob(rnd16(scaled(p.alpha, sacc[e])), mm[r], ll[r], yy[r]);
                            const float tt = pr_ * rnd16(pacc[e]);
                            ds = tt - sg[r] * pr_;
                        }
                        const bool live = FULL || (query >= mykey && query < S);
                        pe[e] = live ? pr_ : 0.f;
                        de[e] = live ? ds : 0.f;
                    }
                }
            };
            if (full) elems(std::true_type{});           // no masks on blocks wholly past the diagonal
            else elems(std::false_type{});
            prod_tr<DT>(vacc, Gs + bf * kTileB, 32 * qb, pack8(pe), pack8(pe + 8), lane);
            prod_tr<DT>(kacc, Qs + bf * kTileB, 32 * qb, pack8(de), pack8(de + 8), lane);
        };
        // tiles [a, b), tile a in LDS and published.  The two blocks are one piece of code, and there are two call sites
        // and not three: a workgroup meets most of its instructions once, coming from memory (51 -> 36 KB of them; 777
        // positions, 16 heads of 128, in parts: 27.1 -> 24.8 us).
        auto run_tiles = [&](int a, int b) __attribute__((always_inline)) {
            for (int iq = a; iq < b; iq++) {
                if (iq + 1 < niq) fetch(iq + 1);
#pragma unroll 1
                for (int qb = qh; qb < (KR == 128 ? 2 : qh + 1); qb++) block(iq, qb);
                if (iq + 1 < niq) land(iq + 1);
                tile_sync<DMA>();
            }
        };

        fetch(iq0);
        land(iq0);
        if constexpr (DMA) {
            // the key and value rows into the second (and third) buffers, idle until the first tile is worked on
#pragma unroll
            for (int t = 0; t < KR / kTileRows; t++) {
                const int64_t off = hoff - shift + (int64_t)(c00 + t * kTileRows) * ld;
                tq.load(tm, gp(p.k) + off, S - (c00 + t * kTileRows), Qs + (1 + t) * kTileB);
                tg.load(tm, gp(p.v) + off, S - (c00 + t * kTileRows), Gs + (1 + t) * kTileB);
            }
            zero_pads(smem, 2 * BUFS * kTileB / kRowB, (Dh + shift + 7) >> 3);
        }
        tile_sync<DMA>();
        if constexpr (DMA) {
            frags_from_tile<KS>(kf, Qs + (1 + (kb >> 1)) * kTileB, (kb & 1) * 32 + l32, Dh, lh, shift);
            frags_from_tile<KS>(vf, Gs + (1 + (kb >> 1)) * kTileB, (kb & 1) * 32 + l32, Dh, lh, shift);
            __syncthreads();                      // every wave holds its fragments: the buffers take query tiles now
        }
        // The tiles that hold the diagonal (two: 128 keys) and a ragged last tile run block by block.  The tiles
        // between them, whose 32-query blocks are whole and past the diagonal for every wave, run as a pipeline
        // (fast arithmetic, tiles loaded straight into LDS): while the vector unit forms P and dS of block b, the
        // matrix unit forms S and dP of block b + 1 and adds block b - 1 to dV and dK.  A wave has its SIMD to
        // itself here, so nothing else would fill the one unit while the other works.
        const int iqB = SPLIT && z > 0 ? iq0 : iq0 + 2, iqE = SPLIT ? min(niq, S / kTileRows) : S / kTileRows;
        const bool pipe = FAST && DMA && KR == 128 && iqE > iqB;
        run_tiles(iq0, pipe ? iqB : niq);
        if (pipe) {
            if constexpr (FAST && DMA && KR == 128) {
                const int a4 = (lane >> 2) & 3, b4 = lane & 3, n16 = (lane >> 4) & 1;
                const int colb = 16 * n16 + 4 * b4;
                // blocks alternate between two register sets: SP = the S and dP accumulators (formed in one
                // step, consumed in the next), PD = the packed P and dS of a block (likewise)
                float16_t SPs[2], SPp[2];
                half8_t PD[2][4];                               // P rows 0..15, P rows 16..31, dS likewise
                half8_t xs[KS], xp[KS], xt[2][DT];
                float4_t yy, sg;
                // S1: the fragment reads of k step t of block (tile q1 / g1, qb1)
                auto x_read = [&](auto t_c, const unsigned char *q1, const unsigned char *g1, int qb1) __attribute__((always_inline)) {
                    constexpr int t = decltype(t_c)::value;
                    const int row = 32 * qb1 + l32, o = row * kRowB + (((2 * t + lh) ^ gsw(row)) << 4);
                    xs[t] = *reinterpret_cast<const half8_t *>(q1 + o);
                    xp[t] = *reinterpret_cast<const half8_t *>(g1 + o);
                };
                // S3: the 2 DT transposing reads of group g = 2 which + kk (which: 0 dV from the dO tile, 1 dK from
                // the Q tile; kk: rows 0..15 or 16..31 of the block), and MFMA j = g DT + dt
                auto t_read = [&](auto g_c, const unsigned char *q3, const unsigned char *g3, int qb3) __attribute__((always_inline)) {
                    constexpr int g = decltype(g_c)::value, which = g >> 1, kk = g & 1;
                    const unsigned char *tile = which ? q3 : g3;
                    const int r1 = 32 * qb3 + 16 * kk + 4 * lh + a4, r2 = r1 + 8;
                    const unsigned char *p1 = tile + r1 * kRowB + ((colb & 4) << 1);
                    const unsigned char *p2 = tile + r2 * kRowB + ((colb & 4) << 1);
                    const int g1_ = gsw(r1), g2_ = gsw(r2);
#pragma unroll
                    for (int dt = 0; dt < DT; dt++) {
                        const int c = (32 * dt + colb) >> 3;
                        xt[g & 1][dt] = as_h8(lds_read_tr(p1 + ((c ^ g1_) << 4)), lds_read_tr(p2 + ((c ^ g2_) << 4)));
                    }
                };
                constexpr int NQ = 32, NM = 2 * KS + 4 * DT;     // quarter pieces of S2 and MFMAs of a step
                // One step.  PAR: parity of the block in S2 (its qb).  S1 forms block (tile1, qb = PAR ^ 1) into
                // set PAR ^ 1, S2 turns set PAR into PD[PAR], S3 adds PD[PAR ^ 1] (block tile3, qb = PAR ^ 1).
                auto step = [&](auto par_c, auto has1_c, auto has3_c, int buf1, int buf2, int buf3) __attribute__((always_inline)) {
                    constexpr int PAR = decltype(par_c)::value, OTH = PAR ^ 1;
                    constexpr bool HAS1 = decltype(has1_c)::value, HAS3 = decltype(has3_c)::value;
                    const unsigned char *q1 = Qs + buf1 * kTileB, *g1 = Gs + buf1 * kTileB;
                    const unsigned char *q3 = Qs + buf3 * kTileB, *g3 = Gs + buf3 * kTileB;
                    const float *stc = St + buf2 * 256;
                    const float16_t &sC = SPs[PAR], &pC = SPp[PAR];
                    // S2 in 32 quarter pieces (8 pairs of elements x 4): the roundings S16 and dP16; the exponentials;
                    // dS; the packed results.  The same operations on the same values as the block-by-block form.
                    half2v_t s2, d2;
                    float pr2[2], ds2[2];
                    auto valu = [&](auto j_c) __attribute__((always_inline)) {
                        constexpr int j = decltype(j_c)::value, pc = j >> 2, qr = j & 3, q = pc >> 1, hf = pc & 1, e0 = 4 * q + 2 * hf;
                        if constexpr (qr == 0) {
                            if constexpr (hf == 0) {
                                const int qi = 32 * PAR + 8 * q + 4 * lh;
                                yy = *reinterpret_cast<const float4_t *>(stc + 2 * 64 + qi);
                                sg = *reinterpret_cast<const float4_t *>(stc + 3 * 64 + qi);
                            }
                            s2 = cvt_pk(scaled(p.alpha, sC[e0]), scaled(p.alpha, sC[e0 + 1]));
                            d2 = cvt_pk(pC[e0], pC[e0 + 1]);
                        } else if constexpr (qr == 1) {
                            pr2[0] = exp2_mix(s2[0], yy[2 * hf]);
                            pr2[1] = exp2_mix(s2[1], yy[2 * hf + 1]);
                        } else if constexpr (qr == 2) {
                            ds2[0] = __builtin_fmaf((float)d2[0], pr2[0], -(sg[2 * hf] * pr2[0]));
                            ds2[1] = __builtin_fmaf((float)d2[1], pr2[1], -(sg[2 * hf + 1] * pr2[1]));
                        } else {
                            half2v_t pn = cvt_pk(pr2[0], pr2[1]), dn = cvt_pk(ds2[0], ds2[1]);
                            // the values are used a step later; without a use here the compiler moves the whole piece there
                            asm volatile("" : "+v"(pn), "+v"(dn));
                            PD[PAR][e0 >> 3][e0 & 7] = pn[0];
                            PD[PAR][e0 >> 3][(e0 & 7) + 1] = pn[1];
                            PD[PAR][2 + (e0 >> 3)][e0 & 7] = dn[0];
                            PD[PAR][2 + (e0 >> 3)][(e0 & 7) + 1] = dn[1];
                        }
                    };
                    if constexpr (HAS1) {
                        x_read(std::integral_constant<int, 0>{}, q1, g1, OTH);
#pragma unroll
                        for (int r = 0; r < 16; r++) {
                            SPs[OTH][r] = 0.f;
                            SPp[OTH][r] = 0.f;
                        }
                    }
                    if constexpr (HAS3) {
                        t_read(std::integral_constant<int, 0>{}, q3, g3, OTH);
                        t_read(std::integral_constant<int, 1>{}, q3, g3, OTH);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    // One MFMA, its share of the 32 quarter pieces, a scheduling barrier: the matrix unit takes 32
                    // cycles per MFMA and a second one issued behind it stalls the wave -- and with it the vector
                    // instructions behind that -- until the first is through.
                    auto slot_end = [&](auto m_c) __attribute__((always_inline)) {
                        constexpr int m = decltype(m_c)::value;
                        __builtin_amdgcn_sched_barrier(0);
                        static_for<m * NQ / NM, (m + 1) * NQ / NM>([&](auto j_c) __attribute__((always_inline)) { valu(j_c); });
                        __builtin_amdgcn_sched_barrier(0);
                    };
                    static_for<0, KS>([&](auto t_c) __attribute__((always_inline)) {
                        constexpr int t = decltype(t_c)::value;
                        constexpr int j0 = t * 4 * DT / KS, j1 = (t + 1) * 4 * DT / KS, m0 = 2 * t + j0;
                        if constexpr (HAS1) SPs[OTH] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xs[t], kf[t], SPs[OTH], 0, 0, 0);
                        slot_end(std::integral_constant<int, m0>{});
                        if constexpr (HAS1) {
                            SPp[OTH] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xp[t], vf[t], SPp[OTH], 0, 0, 0);
                            if constexpr (t + 1 < KS) x_read(std::integral_constant<int, t + 1>{}, q1, g1, OTH);
                        }
                        slot_end(std::integral_constant<int, m0 + 1>{});
                        static_for<j0, j1>([&](auto j_c) __attribute__((always_inline)) {
                            constexpr int j = decltype(j_c)::value, g = j / DT, dt = j % DT, which = g >> 1, kk = g & 1;
                            if constexpr (HAS3) {
                                const half8_t y = PD[OTH][2 * which + kk];
                                if constexpr (which)
                                    kacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xt[g & 1][dt], y, kacc[dt], 0, 0, 0);
                                else
                                    vacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xt[g & 1][dt], y, vacc[dt], 0, 0, 0);
                                // the reads of group g + 2 (two register sets, g & 1) once the last MFMA of group g is out
                                if constexpr (dt == DT - 1 && g + 2 < 4) t_read(std::integral_constant<int, g + 2>{}, q3, g3, OTH);
                            }
                            slot_end(std::integral_constant<int, 2 * t + 2 + j>{});
                        });
                    });
                };
                const std::integral_constant<int, 0> par0;
                const std::integral_constant<int, 1> par1;
                // the first and the last step stand outside the loop, so that the loop holds one form of each step
                // A tile is fetched two steps before its first use and waited for one step before it (the barrier
                // after every second step), so the latency of the loads has a whole step to pass.
                if (iqB + 1 < niq) fetch(iqB + 1);
                SPs[0] = prod_direct<KS, false>(Qs + buf_of(iqB) * kTileB, 0, kf, l32, lh);
                SPp[0] = prod_direct<KS, false>(Gs + buf_of(iqB) * kTileB, 0, vf, l32, lh);
                {
                    const int bc = buf_of(iqB);
                    step(par0, std::true_type{}, std::false_type{}, bc, bc, bc);       // S1 (iqB, 1), S2 (iqB, 0)
                    tile_sync<DMA>();
                }
                for (int iq = iqB; iq + 1 < iqE; iq++) {
                    const int bc = buf_of(iq), bn = buf_of(iq + 1);
                    // step (iq, 1): S1 (iq + 1, 0), S2 (iq, 1), S3 (iq, 0); tile iq + 2 takes the buffer of tile
                    // iq - 1, which the step before was the last to read
                    if (iq + 2 < niq) fetch(iq + 2);
                    step(par1, std::true_type{}, std::true_type{}, bn, bc, bc);
                    // step (iq + 1, 0): S1 (iq + 1, 1), S2 (iq + 1, 0), S3 (iq, 1)
                    step(par0, std::true_type{}, std::true_type{}, bn, bn, bc);
                    tile_sync<DMA>();
                }
                {
                    const int bc = buf_of(iqE - 1);
                    step(par1, std::false_type{}, std::true_type{}, bc, bc, bc);       // S2 (iqE - 1, 1), S3 (iqE - 1, 0)
                }
                prod_tr<DT>(vacc, Gs + buf_of(iqE - 1) * kTileB, 32, PD[1][0], PD[1][1], lane);
                prod_tr<DT>(kacc, Qs + buf_of(iqE - 1) * kTileB, 32, PD[1][2], PD[1][3], lane);
            }
            run_tiles(iqE, niq);
        }
        if constexpr (SPLIT) {
            if (mykey < S) {
                const int64_t plane = (int64_t)p.H * S * Dh;
                float *krow = p.part + z * 2 * plane + ((int64_t)h * S + mykey) * Dh, *vrow = krow + plane;
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int d0 = 32 * dt + 8 * q + 4 * lh - shift;
                        if (d0 >= 0 && d0 < Dh) {
                            *reinterpret_cast<float4_t *>(krow + d0) =
                                float4_t{kacc[dt][4 * q], kacc[dt][4 * q + 1], kacc[dt][4 * q + 2], kacc[dt][4 * q + 3]};
                            *reinterpret_cast<float4_t *>(vrow + d0) =
                                float4_t{vacc[dt][4 * q], vacc[dt][4 * q + 1], vacc[dt][4 * q + 2], vacc[dt][4 * q + 3]};
                        }
                    }
            }
            return;
        }
        if constexpr (KR == 64) {
            // the sums over the second 32 queries of every tile onto those over the first
            float *x = reinterpret_cast<float *>(smem) + kb * 64 + lane;
            if (qh == 1) {
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        x[(dt * 16 + r) * 128] = kacc[dt][r];
                        x[((DT + dt) * 16 + r) * 128] = vacc[dt][r];
                    }
            }
            __syncthreads();
            if (qh == 0) {
#pragma unroll
                for (int dt = 0; dt < DT; dt++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        kacc[dt][r] += x[(dt * 16 + r) * 128];
                        vacc[dt][r] += x[((DT + dt) * 16 + r) * 128];
                    }
            }
        }
        const bool mine = qh == 0, staged_v = DMA && !p.acc_dv, staged_k = DMA && !p.acc_dk;
        if (staged_v || staged_k) {
            __syncthreads();                              // the last products have read their tiles
            if (staged_k && mine) stage_rows<DT>(Qs, kacc, kb * 32 + l32, lh, p.alpha);
            if (staged_v && mine) stage_rows<DT>(Gs, vacc, kb * 32 + l32, lh, 1.0f);
            __syncthreads();
            const int64_t off = (int64_t)c00 * ld + hoff - shift;
            if (staged_k) write_rows(Qs, p.dk + off, ld, min(KR, S - c00), Dh, shift, threadIdx.x, kNT);
            if (staged_v) write_rows(Gs, p.dv + off, ld, min(KR, S - c00), Dh, shift, threadIdx.x, kNT);
        }
        if (mine && mykey < S && !(staged_v && staged_k)) {
            half_t *krow = p.dk + (int64_t)mykey * ld + hoff, *vrow = p.dv + (int64_t)mykey * ld + hoff;
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int d0 = 32 * dt + 8 * q + 4 * lh - shift;
                    if (d0 >= 0 && d0 < Dh) {
                        if (!staged_v)
                            store_row4(vrow + d0, vacc[dt][4 * q], vacc[dt][4 * q + 1], vacc[dt][4 * q + 2],
                                       vacc[dt][4 * q + 3], 1.0f, p.acc_dv);
                        if (!staged_k)
                            store_row4(krow + d0, kacc[dt][4 * q], kacc[dt][4 * q + 1], kacc[dt][4 * q + 2],
                                       kacc[dt][4 * q + 3], p.alpha, p.acc_dk);
                    }
                }
        }
    }
}

// dK and dV from the sums of their parts, added in order; four columns per lane, blockIdx.y = 0 dK, 1 dV
__global__ void __launch_bounds__(256) attn_bwd_dkv_sum_kernel(AttnArgs p)
{
    const int per_row = p.Dh / 4;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, plane = (int64_t)p.H * p.S * p.Dh;
    if (i >= plane / 4) return;
    const int64_t row = i / per_row;                                    // h * S + key
    const int h = (int)(row / p.S), key = (int)(row - (int64_t)h * p.S), d = (int)(i - row * per_row) * 4;
    const int tiles = (p.S + kTileRows - 1) / kTileRows - key / kBM * (kBM / kTileRows), parts = (tiles + p.per - 1) / p.per;
    const float *src = p.part + blockIdx.y * plane + 4 * i;
    float4_t a = *reinterpret_cast<const float4_t *>(src);
    for (int z = 1; z < parts; z++) a += *reinterpret_cast<const float4_t *>(src + z * 2 * plane);
    half_t *dst = (blockIdx.y ? p.dv : p.dk) + key * p.ld + (int64_t)h * p.Dh + d;
    store_row4(dst, a[0], a[1], a[2], a[3], blockIdx.y ? 1.0f : p.alpha, blockIdx.y ? p.acc_dv : p.acc_dk);
}

// A workgroup of the dK / dV kernel walks all query tiles from its keys on, 1.4 us each behind some 10 us of start, and
// a short sequence has few workgroups for it (1000 positions of 4 heads: 32 of up to 16 tiles, on 256 CUs).  There the
// query tiles of 128 keys go to several workgroups, as many as the device has room for, whose fp32 sums a second launch of
// 4.6 to 6.6 us adds up.  Against one walk with 64 keys (few_keys: half the work per tile) a part has to be at least 8 tiles
// shorter than the walk: adjoint with 64 keys -> parts, us, 449 positions, 8 heads of 64 (6 tiles shorter) 27.7 -> 28.5; 611, 4 of
// 64 (8) 29.2 -> 27.8; 1000, 4 of 100 (14) 52 -> 44.6.  What it is weighed against where it runs is the walk of attention_short.hip,
// which takes all of those and leaves parts the longest sequences of few heads: attention_short_dkv_takes.  split = 1: not.  The
// exact arithmetic has no parts.
struct DkvParts {
    int split, per;
};
DkvParts dkv_parts(int64_t S, int64_t H, bool exact)
{
    const int64_t groups = (S + kBM - 1) / kBM * H, tiles = (S + kTileRows - 1) / kTileRows;
    int64_t split = std::min<int64_t>(device_cus() / groups, 8);
    if (exact || split < 2) return {1, (int)tiles};
    const int64_t per = std::max<int64_t>(2, (tiles + split - 1) / split);
    if (tiles - per < 8) return {1, (int)tiles};
    return {(int)((tiles + per - 1) / per), (int)per};
}
size_t stats_part_bytes(int64_t S, int64_t H) { return ((size_t)(2 * S * H) * sizeof(float) + 15) / 16 * 16; }
size_t parts_bytes(const DkvParts &parts, int64_t S, int64_t H, int64_t Dh)
{
    return (size_t)parts.split * 2 * (size_t)H * (size_t)S * (size_t)Dh * sizeof(float);
}

constexpr size_t dkv_smem(int keys) { return (2 * kTileB + 4 * 64 * sizeof(float)) * dkv_bufs(keys); }

template <class K>
int set_smem(K kern, size_t bytes)
{
    CACTI_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
    return 0;
}

// Which arithmetic the kernels are launched with (AttnMath).  Measured at 32 heads x 2048 x 100 on MI355X, in a hot loop:
// forward 64 us / adjoint 145 us with the fast form, 101 / 251 us with the exact one, which has no in-wave pipelines, no short
// form of sigma and no parts; the two differ by 3e-5 .. 4e-5 relative L2 in O, dQ, dK, dV, and O, dQ, dK, dV of the fast form
// agree with the CPU restatement of the reference to 4.9e-5 .. 7.1e-5.
std::atomic<int> g_exact{0};             // cacti_hip_attention_set_exact: launch the exactly rounded forms

// Query rows per workgroup of the forward and the dQ kernel, 64 or 128, where attention_short.hip does not take the call.  A
// workgroup has a CU to itself and walks its keys
// 128 at a time; with 64 rows two waves share a tile's keys, so a step takes less time (one head of 128: 2.1 us against 2.85
// forward) and there are twice as many workgroups, each of which reads all keys.  Worth it until they need a third round
// over the CUs: 128 -> 64 rows, us, forward and adjoint (its dQ alone), 1100 positions, 20 heads of 64 (360 workgroups) 30.0 -> 25.6
// and 56 -> 50; 1531, 16 of 128 (384) 42.9 -> 34.7 and 93 -> 78; 1984, 16 of 128 (496) 54.2 -> 47.8 and 117 -> 107; 4096, 8 of 128
// (512) 100 -> 84 and 199 -> 184; 1300, 26 of 64 (546) 33.1 -> 41.6 and 64 -> 65; 1422, 24 of 100 (552) 40.8 -> 49.6 and 100 -> 95;
// 2048, 32 of 100 (1024) 68 -> 95 and 156 -> 168.  Exact arithmetic: 1531, 16 of 128 70.0 -> 45.4 and 143 -> 108; 1000, 26 of 64
// (416) 45.6 -> 34.1 and 89 -> 70.  Up to 128 positions there is a step or two either way.
// The forward kernel's second round is short only if there are long sequences in the first.  Up to 1024 positions it is left heads
// to 64 between 3/2 and 2 workgroups per CU, where the default arithmetic is as good either way from 770 positions on (1000, 25 of
// 64 28.2 -> 27.0; 832, 32 24.6 -> 24.3; 896, 32 25.7 -> 26.0; 1024, 28 27.8 -> 28.4) and better with 128 rows below (768, 36 of 64
// 23.4 -> 25.1; 640, 40 21.2 -> 22.6; 450, 52 19.1 -> 21.9).
int query_rows(int64_t S, int64_t H, bool forward, bool fast)
{
    return S > (forward && fast ? 1024 : 128) && (S + 63) / 64 * H <= 2 * (int64_t)device_cus() ? 64 : 128;
}

// Whether the dK / dV kernel takes 64 keys per workgroup instead of 128: its workgroups then walk the same query tiles with
// half of the work in each (two waves to 32 keys), but without the in-wave pipeline.  Adjoint with 128 -> 64 keys, us: 1531
// positions, 16 heads of 128 (384 workgroups) 86 -> 75; 2048, 16 of 128
// (512) 113 -> 108; 1051, 32 of 100 (544) 80 -> 87.  Heads to 64 leave registers for two workgroups per CU: 2048, 16 of 64
// 94 -> 78; 2048, 32 of 64 (1024) 125 -> 117.  Parts of the query tiles, where there are any, are better (dkv_parts).
bool few_keys(const AttnArgs &p, bool narrow)
{
    const int64_t tiles = (p.S + kTileRows - 1) / kTileRows;
    return p.S > 128 && tiles * p.H <= (narrow ? 4 : 2) * (int64_t)device_cus() && p.split < 2;
}

template <int KS, int DT, bool FAST, bool DMA>
int launch_fwd(const AttnArgs &p, hipStream_t st)
{
    static DeviceOnce ready;
    if (!ready.fresh()) {
        int rc = set_smem(attn_fwd_kernel<KS, DT, FAST, DMA, 128>, kQmSmem);
        if (rc) return rc;
        if constexpr (DMA)
            if ((rc = set_smem(attn_fwd_kernel<KS, DT, FAST, DMA, 64>, kQmSmem))) return rc;
        ready.mark();
    }
    const int rows = DMA ? query_rows(p.S, p.H, true, FAST) : 128, nqt = (p.S + rows - 1) / rows;
    const dim3 grid((unsigned)(nqt * p.H));
    if constexpr (DMA)
        if (rows == 64) hipLaunchKernelGGL((attn_fwd_kernel<KS, DT, FAST, DMA, 64>), grid, dim3(kNT2), kQmSmem, st, p);
    if (rows == 128) hipLaunchKernelGGL((attn_fwd_kernel<KS, DT, FAST, DMA, 128>), grid, dim3(kNT2), kQmSmem, st, p);
    return launch_status("attention_fwd");
}

template <int KS, int DT, bool FAST, bool DMA>
int launch_dq(const AttnArgs &p, hipStream_t st)
{
    static DeviceOnce ready;
    if (!ready.fresh()) {
        int rc = set_smem(attn_bwd_dq_kernel<KS, DT, FAST, DMA, 128>, kQmSmem);
        if (rc) return rc;
        if constexpr (DMA)
            if ((rc = set_smem(attn_bwd_dq_kernel<KS, DT, FAST, DMA, 64>, kQmSmem))) return rc;
        ready.mark();
    }
    const int rows = DMA ? query_rows(p.S, p.H, false, FAST) : 128;
    const dim3 grid((unsigned)((p.S + rows - 1) / rows * p.H));
    if constexpr (DMA)
        if (rows == 64) hipLaunchKernelGGL((attn_bwd_dq_kernel<KS, DT, FAST, DMA, 64>), grid, dim3(kNT2), kQmSmem, st, p);
    if (rows == 128) hipLaunchKernelGGL((attn_bwd_dq_kernel<KS, DT, FAST, DMA, 128>), grid, dim3(kNT2), kQmSmem, st, p);
    return launch_status("attention_bwd_dq");
}

template <int KS, int DT, bool FAST, bool DMA>
int launch_dkv(const AttnArgs &p, hipStream_t st)
{
    constexpr bool PARTS = FAST && DMA;
    static DeviceOnce ready;
    if (!ready.fresh()) {
        int rc;
        if ((rc = set_smem(attn_bwd_dkv_kernel<KS, DT, FAST, DMA, false, 128>, dkv_smem(128)))) return rc;
        if constexpr (DMA)
            if ((rc = set_smem(attn_bwd_dkv_kernel<KS, DT, FAST, DMA, false, 64>, dkv_smem(64)))) return rc;
        if constexpr (PARTS)
            if ((rc = set_smem(attn_bwd_dkv_kernel<KS, DT, FAST, DMA, true, 128>, dkv_smem(128)))) return rc;
        ready.mark();
    }
    const int nqt = (p.S + kBM - 1) / kBM;
    if constexpr (DMA)
        if (few_keys(p, KS == 4)) {
            hipLaunchKernelGGL((attn_bwd_dkv_kernel<KS, DT, FAST, DMA, false, 64>), dim3((unsigned)((p.S + 63) / 64 * p.H)), dim3(kNT),
                               dkv_smem(64), st, p);
            return launch_status("attention_bwd_dkv");
        }
    if constexpr (PARTS)
        if (p.split > 1) {
            hipLaunchKernelGGL((attn_bwd_dkv_kernel<KS, DT, FAST, DMA, true, 128>), dim3((unsigned)(nqt * p.split * p.H)), dim3(kNT),
                               dkv_smem(128), st, p);
            const int64_t lanes = (int64_t)p.H * p.S * (p.Dh / 4);
            hipLaunchKernelGGL(attn_bwd_dkv_sum_kernel, dim3((unsigned)((lanes + 255) / 256), 2), dim3(256), 0, st, p);
            return launch_status("attention_bwd_dkv");
        }
    hipLaunchKernelGGL((attn_bwd_dkv_kernel<KS, DT, FAST, DMA, false, 128>), dim3((unsigned)(nqt * p.H)), dim3(kNT), dkv_smem(128), st, p);
    return launch_status("attention_bwd_dkv");
}

// Whether the tiles of these tensors can be loaded straight into LDS: 16-byte aligned tensors and rows, and
// every head's window (from the 16-byte boundary at or below its start, whole 16-byte chunks) inside its row.
// *span = the window positions a head can occupy (Dh + the largest shift).
bool direct_tiles(int64_t H, int64_t Dh, int64_t ld, std::initializer_list<const void *> tensors, int64_t *span)
{
    *span = Dh;
    if (ld % 8 != 0) return false;
    for (const void *t : tensors)
        if (!aligned(t, 16)) return false;
    int64_t most = 0;
    for (int64_t h = 0; h < H; h++) {
        const int64_t shift = (h * Dh) & 7, start = h * Dh - shift, chunks = (Dh + shift + 7) / 8;
        if (start + 8 * chunks > ld || 8 * chunks > kDP) return false;
        most = std::max(most, Dh + shift);
    }
    *span = most;
    return true;
}

// the instantiation by the window span (16 KS and 32 DT positions must cover it), the arithmetic and the loader
template <template <int, int, bool, bool> class L>
int dispatch(int64_t span, bool exact, bool dma, const AttnArgs &p, hipStream_t st)
{
    auto by_size = [&](auto fast_c, auto dma_c) {
        constexpr bool F = decltype(fast_c)::value, D = decltype(dma_c)::value;
        if (span <= 64) return L<4, 2, F, D>::run(p, st);
        if (span <= 112) return L<7, 4, F, D>::run(p, st);
        return L<8, 4, F, D>::run(p, st);
    };
    if (exact) return dma ? by_size(std::false_type{}, std::true_type{}) : by_size(std::false_type{}, std::false_type{});
    return dma ? by_size(std::true_type{}, std::true_type{}) : by_size(std::true_type{}, std::false_type{});
}
template <int KS, int DT, bool F, bool D> struct Fwd { static int run(const AttnArgs &p, hipStream_t st) { return launch_fwd<KS, DT, F, D>(p, st); } };
template <int KS, int DT, bool F, bool D> struct BwdDq { static int run(const AttnArgs &p, hipStream_t st) { return launch_dq<KS, DT, F, D>(p, st); } };
template <int KS, int DT, bool F, bool D> struct BwdDkv { static int run(const AttnArgs &p, hipStream_t st) { return launch_dkv<KS, DT, F, D>(p, st); } };

int check_shape(const char *who, int64_t S, int64_t H, int64_t Dh, int64_t ld)
{
    CACTI_REQUIRE(S > 0 && H > 0 && Dh > 0, CACTI_E_INVALID, "%s: empty shape", who);
    CACTI_REQUIRE(Dh % 4 == 0 && Dh <= kDP, CACTI_E_NOTIMPL, "%s: need Dh %% 4 == 0 and Dh <= %d (Dh=%lld)", who, kDP,
                  (long long)Dh);
    CACTI_REQUIRE(ld >= H * Dh && ld % 4 == 0, CACTI_E_INVALID, "%s: row stride %lld must be a multiple of 4 and >= H*Dh",
                  who, (long long)ld);
    CACTI_REQUIRE(S <= (1 << 24) && S * H < ((int64_t)1 << 31) / 2, CACTI_E_NOTIMPL, "%s: S = %lld is too large", who,
                  (long long)S);
    // the tile loaders keep (row within a tile) * ld + column as a 32-bit offset
    CACTI_REQUIRE(ld <= ((int64_t)1 << 26), CACTI_E_NOTIMPL, "%s: row stride %lld is beyond the 2^26 elements the "
                  "tile loaders address", who, (long long)ld);
    return 0;
}

}  // namespace

CACTI_API int cacti_hip_attention_set_exact(int on)
{
    g_exact.store(on ? 1 : 0, std::memory_order_relaxed);
    return 0;
}

CACTI_API size_t cacti_hip_attention_stats_bytes(int64_t S, int64_t H)
{
    return (S > 0 && H > 0) ? (size_t)(2 * S * H) * sizeof(float) : 0;
}

CACTI_API size_t cacti_hip_attention_bwd_workspace(int64_t S, int64_t H)
{
    return (S > 0 && H > 0) ? (size_t)(2 * S * H) * sizeof(float) : 0;
}

static int attention_fwd(int64_t S, int64_t H, int64_t Dh, float alpha, const void *q, const void *k, const void *v, int64_t ld, void *o,
                         void *stats, bool exact, bool windows, hipStream_t st)
{
    int rc = check_shape("attention_fwd", S, H, Dh, ld);
    if (rc) return rc;
    CACTI_REQUIRE(q && k && v && o && stats, CACTI_E_INVALID, "attention_fwd: null pointer");
    CACTI_REQUIRE(aligned(q, 8) && aligned(k, 8) && aligned(v, 8) && aligned(o, 8) && aligned(stats, 4),
                  CACTI_E_INVALID, "attention_fwd: tensors must be 8-byte aligned");
    AttnArgs p = {};
    p.S = (int)S; p.H = (int)H; p.Dh = (int)Dh; p.ld = ld; p.alpha = alpha;
    p.q = (const half_t *)q; p.k = (const half_t *)k; p.v = (const half_t *)v;
    p.out = (half_t *)o;
    p.m = (float *)stats;
    p.l = p.m + S * H;
    int64_t span = Dh;
    const bool dma = (windows || Dh % 8 == 0) && direct_tiles(H, Dh, ld, {q, k, v, o}, &span);
    if (dma && attention_short_fwd_takes(S, H, span)) return attention_short_fwd(p, span, exact, st);
    return dispatch<Fwd>(span, exact, dma, p, st);
}

CACTI_API int cacti_hip_attention_fwd(int64_t S, int64_t H, int64_t Dh, float alpha, const void *q, const void *k,
                                      const void *v, int64_t ld, void *o, void *stats, void *stream)
{
    return attention_fwd(S, H, Dh, alpha, q, k, v, ld, o, stats, g_exact.load(std::memory_order_relaxed) != 0, true, (hipStream_t)stream);
}

namespace cacti {

// For the cached forward pass: the exactly rounded form whatever the process-wide setting, and every head by its own
// elements alone, as with scores, softmax and P V apart.  Heads that start between 16-byte boundaries then come through
// registers: a window of 16-byte pieces holds 4 elements of the next head, and a key of -infinity there (a score of
// -infinity, a probability of 0 in its own head) would make this head's scores NaN.
int attention_fwd_exact(int64_t S, int64_t H, int64_t Dh, float alpha, const void *q, const void *k, const void *v, int64_t ld, void *o,
                        void *stats, hipStream_t st)
{
    return attention_fwd(S, H, Dh, alpha, q, k, v, ld, o, stats, true, false, st);
}

}  // namespace cacti

CACTI_API size_t cacti_hip_attention_bwd_workspace_best(int64_t S, int64_t H, int64_t Dh)
{
    if (S <= 0 || H <= 0 || Dh <= 0 || Dh > kDP) return cacti_hip_attention_bwd_workspace(S, H);
    const DkvParts parts = dkv_parts(S, H, g_exact.load(std::memory_order_relaxed) != 0);
    if (parts.split < 2) return cacti_hip_attention_bwd_workspace(S, H);
    return stats_part_bytes(S, H) + parts_bytes(parts, S, H, Dh);
}

CACTI_API size_t cacti_hip_attention_bwd_workspace_used(int64_t S, int64_t H, int64_t Dh, int64_t ld)
{
    const size_t least = cacti_hip_attention_bwd_workspace(S, H);
    if (S <= 0 || H <= 0 || Dh <= 0 || Dh > kDP) return least;
    const DkvParts parts = dkv_parts(S, H, g_exact.load(std::memory_order_relaxed) != 0);
    int64_t span;
    // (parts are of tiles straight from memory, and with those a walk over all queries is the better form of most shapes)
    if (parts.split < 2 || !direct_tiles(H, Dh, ld, {}, &span) || attention_short_dkv_takes(S, H, span, parts.per)) return least;
    return cacti_hip_attention_bwd_workspace_best(S, H, Dh);
}

CACTI_API int cacti_hip_attention_bwd(int64_t S, int64_t H, int64_t Dh, float alpha, const void *q, const void *k,
                                      const void *v, const void *o, const void *dO, int64_t ld, const void *stats,
                                      void *dq, int dq_acc, void *dk, int dk_acc, void *dv, int dv_acc,
                                      void *workspace, size_t workspace_bytes, void *stream)
{
    int rc = check_shape("attention_bwd", S, H, Dh, ld);
    if (rc) return rc;
    CACTI_REQUIRE(q && k && v && dO && stats && dq && dk && dv && workspace, CACTI_E_INVALID,
                  "attention_bwd: null pointer");
    CACTI_REQUIRE(aligned(q, 8) && aligned(k, 8) && aligned(v, 8) && aligned(dO, 8) && aligned(o, 8) &&
                      aligned(dq, 8) && aligned(dk, 8) && aligned(dv, 8) && aligned(stats, 4) && aligned(workspace, 4),
                  CACTI_E_INVALID, "attention_bwd: tensors must be 8-byte aligned");
    CACTI_REQUIRE(workspace_bytes >= cacti_hip_attention_bwd_workspace(S, H), CACTI_E_INVALID,
                  "attention_bwd: workspace of %zu bytes is smaller than the %zu needed", workspace_bytes,
                  cacti_hip_attention_bwd_workspace(S, H));
    AttnArgs p = {};
    p.S = (int)S; p.H = (int)H; p.Dh = (int)Dh; p.ld = ld; p.alpha = alpha;
    p.q = (const half_t *)q; p.k = (const half_t *)k; p.v = (const half_t *)v;
    p.dO = (const half_t *)dO;
    p.o = (const half_t *)o;
    p.dq = (half_t *)dq; p.dk = (half_t *)dk; p.dv = (half_t *)dv;
    p.acc_dq = dq_acc; p.acc_dk = dk_acc; p.acc_dv = dv_acc;
    p.m = (float *)const_cast<void *>(stats);
    p.l = p.m + S * H;
    p.y = (float *)workspace;
    p.sig = p.y + S * H;
    const bool exact = g_exact.load(std::memory_order_relaxed) != 0;
    const DkvParts parts = dkv_parts(S, H, exact);
    if (parts.split > 1 && aligned(workspace, 16) && workspace_bytes >= stats_part_bytes(S, H) + parts_bytes(parts, S, H, Dh)) {
        p.split = parts.split;
        p.per = parts.per;
        p.part = reinterpret_cast<float *>(static_cast<char *>(workspace) + stats_part_bytes(S, H));
    }
    hipStream_t st = (hipStream_t)stream;
    int64_t span;
    const bool dma = direct_tiles(H, Dh, ld, {q, k, v, dO, o, dq, dk, dv}, &span);     // o may be null: passes
    rc = dma && attention_short_dq_takes(S, H, exact) ? attention_short_dq(p, span, exact, st) : dispatch<BwdDq>(span, exact, dma, p, st);
    if (rc) return rc;
    if (dma && attention_short_dkv_takes(S, H, span, p.split > 1 ? p.per : 0)) return attention_short_dkv(p, span, exact, st);
    return dispatch<BwdDkv>(span, exact, dma, p, st);
}
