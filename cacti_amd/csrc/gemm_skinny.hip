// C[M,N] = f16(alpha * A[M,K] B[N,K]^T) for M <= 4 rows (decoding: one or a few positions against
// a weight matrix).  The product is a stream over B: every byte of the weights is read once and
// used M times, so the kernel is built for HBM, not for the matrix cores.
//
// A workgroup of 64 or 256 lanes owns R = 4 rows of B (4 output columns) and splits K over its lanes
// in 16-byte pieces; a lane issues the loads of its 1 to 5 pieces x 4 rows before it uses the first (a longer row
// takes several such passes),
// accumulates M x 4 fp32 sums with v_dot2_f32_f16 (the scalar form, 3 instructions per product
// with the conversions, made the kernel compute-bound), and the sums are reduced over the wave (cross-lane adds) and
// over the waves (LDS).  N / 4 workgroups: 800 for N = 3200, 8 resident per CU.  A (a few KiB)
// is re-read from L2 by every workgroup.  What a launch costs beyond its bytes at 6 TB/s is some 4 us: start, the first
// loads' latency, the norm and the reductions.
//
// Two fusions keep a decoding step from paying a launch for every small thunk:
//  * NORM: A is not read but formed per workgroup as the RMSNorm of a row x (optionally of the
//    residual sum f16(x + x2), which workgroup 0 also writes out): the lanes' own pieces of the
//    row give the sum of squares (every piece of the row belongs to exactly one lane), one
//    workgroup reduction, then a = f16(w * (x * rinv)).  The RMSNorm kernel sums in fp64 and divides;
//    here the sum is fp32 and rinv a rounded reciprocal, which moves 8 elements of 100,000 to
//    the neighbouring f16.
//  * GATE: two weight matrices share the rows (gate and up projection); the epilogue stores
//    f16(f16(silu(g)) * u) of the two rounded products, as the SiLU-gate kernel computes it.
//  * QKV: one launch covers the query, key and value projections; a workgroup owns two rotation
//    pairs of a head, rotates queries and keys in the epilogue and adds keys and values to the
//    cache rows of the new positions.
#include "gemm_internal.h"

namespace cacti {

namespace {

constexpr int kRows = 4;
constexpr int kMaxNorm = 1024;             // 16-byte pieces of a row that NORM takes (4 waves x 4 pieces per lane)

struct SkinnyArgs {
    int64_t N, K;
    float alpha;
    const half_t *A;         // [M, lda] (plain) or the row source x (NORM)
    int64_t lda;
    const half_t *x2;        // NORM: optional second summand of the row
    const half_t *w;         // NORM: norm weights [K]
    float eps;
    half_t *sum_out;         // NORM with x2: the residual sum [M, lda], written by workgroup 0
    const half_t *B;         // [N, ldb]
    const half_t *B2;        // GATE: the second weight matrix [N, ldb]; QKV: the key projection
    int64_t ldb;
    half_t *C;               // QKV: the rotated queries [M, ldc]
    int64_t ldc;
    // QKV: value projection, position tables (row 0 = the first new position), caches (row 0 = the
    // first new position, pitch ldc), heads
    const half_t *B3;
    const half_t *cos16, *sin16;
    half_t *kc, *vc;
    int H, Dh;
    FastDiv half_head;       // by Dh / 2
    // NORM: with tok, row m of x is row tok[m] of A (the embedding of `vocab` rows); an id out of range raises
    // *status to m + 1 and reads the last row
    const uint16_t *tok;
    int64_t vocab;
    int *status;
    // E_PLAIN: with cand, the largest result of the workgroup's columns, cand[m * workgroups + workgroup] (arg_key)
    uint32_t *cand;
};
enum : int { E_PLAIN = 0, E_GATE = 1, E_QKV = 2 };

// An f16 result and its column (below 65536) as one number that orders as the arg max does: by value, the first
// column of equal values (+0 and -0 are equal), no NaN.
__device__ __forceinline__ uint32_t arg_key(half_t v, int64_t n)
{
    uint16_t b = __builtin_bit_cast(uint16_t, v);
    if ((b & 0x7fff) > 0x7c00) return 0;
    if (b == 0x8000) b = 0;
    const uint32_t o = b & 0x8000 ? (uint16_t)~b : b | 0x8000u;
    return o << 16 | (uint32_t)(0xffff - n);
}

// sum of 8 products, fp32 accumulate: four v_dot2_f32_f16 (no conversions, two products each)
__device__ __forceinline__ float dot8(const half8_t &a, const half8_t &b, float acc)
{
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const half2_t a2 = {a[2 * i], a[2 * i + 1]}, b2 = {b[2 * i], b[2 * i + 1]};
        acc = __builtin_amdgcn_fdot2(a2, b2, acc, false);
    }
    return acc;
}

// W waves split K, kPre pieces per lane and pass.
template <int M, bool NORM, int EPI, int W, int kPre>
__global__ void __launch_bounds__(W * 64)
gemm_skinny_nt_kernel(SkinnyArgs p)
{
    // the argument block in scalar registers at once: field by field where the control flow first wants it, it is several
    // round trips to memory before the weights are requested
    if (NORM)
        asm volatile("" ::"s"(p.N), "s"(p.K), "s"(p.alpha), "s"(p.A), "s"(p.lda), "s"(p.B), "s"(p.ldb), "s"(p.C), "s"(p.ldc),
                     "s"(p.x2), "s"(p.w), "s"(p.eps), "s"(p.sum_out), "s"(p.tok), "s"(p.vocab));
    if (NORM && EPI != E_PLAIN) asm volatile("" ::"s"(p.B2));
    if (EPI == E_QKV)
        asm volatile("" ::"s"(p.B3), "s"(p.cos16), "s"(p.sin16), "s"(p.kc), "s"(p.vc), "s"(p.H), "s"(p.Dh), "s"(p.half_head.m),
                     "s"(p.half_head.shift));
    constexpr int kThreads = W * 64;
    constexpr bool GATE = EPI == E_GATE;
    constexpr int NB = GATE ? 2 : 1;
    __shared__ float part[W][NB * M * kRows];
    __shared__ float scratch[M][W];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int64_t n0 = (int64_t)blockIdx.x * kRows;
    float acc[NB][M][kRows];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int r = 0; r < kRows; r++) acc[b][m][r] = 0.f;
    const half_t *arow[M];
#pragma unroll
    for (int m = 0; m < M; m++) {
        arow[m] = p.A + m * p.lda;
        if (NORM && p.tok) {
            int64_t id = p.tok[m];
            if (id >= p.vocab) {
                if (tid == 0 && blockIdx.x == 0 && blockIdx.y == 0 && p.status) atomicMax(p.status, m + 1);
                id = p.vocab - 1;
            }
            arow[m] = p.A + id * p.lda;
        }
    }
    const int64_t chunks = p.K / 8;
    h8 a[kPre][M], wv[NORM ? kPre : 1], x2v[NORM ? kPre : 1][M];
    // Loads return in order, so with NORM (the whole row in one batch) the row and its norm weights go first, and the norm
    // is worked out while the weights stream (gate and up of 5504 x 2048 10.5 -> 10.0 us; without a norm the row goes last:
    // first it costs 3 % at 3200 x 8640).  They are requested before the weights' addresses are worked out, and the one batch
    // is said to be one: in a loop over batches the compiler moves the first steps of the norm in front of it, i.e. in front
    // of the weights' requests.  With that, q, k, v's cells and angles requested here and the arguments read at once: q, k, v
    // of 2048 8.1 -> 6.9 us, gate and up 10.0 -> 9.6, a head of 32000 x 2048 22.3 -> 20.6; four rows of 3200: q, k, v
    // 52 -> 28, gate and up 57 -> 36, head 142 -> 71.
    if (NORM) {
#pragma unroll
        for (int j = 0; j < kPre; j++) {
            const int64_t cr = j * kThreads + tid, c = cr < chunks ? cr : chunks - 1;
#pragma unroll
            for (int m = 0; m < M; m++) {
                a[j][m] = ld8(arow[m] + c * 8);
                x2v[j][m] = ld8((p.x2 ? p.x2 + m * p.lda : arow[m]) + c * 8);
            }
            wv[j] = ld8(p.w + c * 8);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // rows past N re-read the last row (their sums are dropped)
    const half_t *brow[NB][kRows];
    int64_t col[kRows];
    int dcol[kRows];                                         // QKV: the column inside its head
    if (EPI == E_QKV) {
        // the workgroup owns kRows / 2 consecutive rotation pairs (columns d and d + Dh/2 of a head), the left columns
        // in the first half of its rows; blockIdx.y picks the query, key or value projection
        // (Dh / 2 is even: both pairs are of one head)
        const int hf = p.Dh / 2, head = p.half_head.div(blockIdx.x * (kRows / 2)), d0 = blockIdx.x * (kRows / 2) - head * hf;
        const half_t *Bsel = blockIdx.y == 0 ? p.B : blockIdx.y == 1 ? p.B2 : p.B3;
#pragma unroll
        for (int r = 0; r < kRows; r++) {
            dcol[r] = d0 + r % (kRows / 2) + (r / (kRows / 2)) * hf;
            col[r] = (int64_t)head * p.Dh + dcol[r];
            brow[0][r] = Bsel + col[r] * p.ldb;
        }
    } else {
#pragma unroll
        for (int r = 0; r < kRows; r++) {
            col[r] = n0 + r;
            const int64_t n = n0 + r < p.N ? n0 + r : p.N - 1;
            brow[0][r] = p.B + n * p.ldb;
            if (GATE) brow[NB - 1][r] = p.B2 + n * p.ldb;
        }
    }
    // QKV: what the epilogue needs from memory, lane (m, r); requested with the weights
    const int er = tid % kRows, em = tid / kRows < M ? tid / kRows : M - 1;
    int64_t ecol = 0;
    half_t ecos = 0, esin = 0, ecell = 0;
    for (int64_t base = 0; base < (NORM ? 1 : chunks); base += (int64_t)kPre * kThreads) {
        half8_t b[kPre][NB][kRows];
        // Every load of the batch is issued before the first use, unconditionally (pieces past the row re-read its last
        // piece): a load inside a branch is waited for at the end of the branch.
#pragma unroll
        for (int j = 0; j < kPre; j++) {
            const int64_t cr = base + j * kThreads + tid, c = cr < chunks ? cr : chunks - 1;
#pragma unroll
            for (int q = 0; q < NB; q++)
#pragma unroll
                for (int r = 0; r < kRows; r++)
                    b[j][q][r] = __builtin_nontemporal_load(reinterpret_cast<const half8_t *>(brow[q][r]) + c);
            if (!NORM) {
#pragma unroll
                for (int m = 0; m < M; m++) a[j][m] = ld8(arow[m] + c * 8);
            }
        }
        if (EPI == E_QKV) {
            int d = dcol[0];
            ecol = col[0];
#pragma unroll
            for (int r = 1; r < kRows; r++) {
                d = er == r ? dcol[r] : d;
                ecol = er == r ? col[r] : ecol;
            }
            ecos = p.cos16[em * p.Dh + d];
            esin = p.sin16[em * p.Dh + d];
            ecell = (blockIdx.y == 1 ? p.kc : p.vc)[em * p.ldc + ecol];
        }
        if (NORM) __builtin_amdgcn_sched_barrier(0);
        if (NORM) {
            // the whole row is in this one batch (K <= 8 * kPre * kThreads, seen to by the launcher); one barrier for all rows
            float ss[M];
#pragma unroll
            for (int m = 0; m < M; m++) {
                ss[m] = 0.f;
#pragma unroll
                for (int j = 0; j < kPre; j++) {
                    const int64_t c = base + j * kThreads + tid;
                    if (c < chunks) {
                        if (p.x2) {
#pragma unroll
                            for (int i = 0; i < 8; i++) a[j][m].v[i] = f2h(h2f(a[j][m].v[i]) + h2f(x2v[j][m].v[i]));
                            if (blockIdx.x == 0 && blockIdx.y == 0 && p.sum_out) st8(p.sum_out + m * p.lda + c * 8, a[j][m]);
                        }
#pragma unroll
                        for (int i = 0; i < 8; i++) {
                            const float f = h2f(a[j][m].v[i]);
                            ss[m] += f * f;
                        }
                    }
                }
                ss[m] = wave_sum(ss[m]);
                if (W > 1 && lane == 0) scratch[m][wid] = ss[m];
            }
            if (W > 1) {
                __syncthreads();
#pragma unroll
                for (int m = 0; m < M; m++) {
                    ss[m] = scratch[m][0];
#pragma unroll
                    for (int w = 1; w < W; w++) ss[m] += scratch[m][w];
                }
            }
#pragma unroll
            for (int m = 0; m < M; m++) {
                const float rinv = 1.0f / sqrtf(ss[m] / (float)p.K + p.eps);
#pragma unroll
                for (int j = 0; j < kPre; j++) {
                    const int64_t c = base + j * kThreads + tid;
                    if (c < chunks) {
#pragma unroll
                        for (int i = 0; i < 8; i++) a[j][m].v[i] = f2h(h2f(wv[j].v[i]) * (h2f(a[j][m].v[i]) * rinv));
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < kPre; j++) {
            const int64_t c = base + j * kThreads + tid;
            if (c < chunks) {
#pragma unroll
                for (int m = 0; m < M; m++) {
                    half8_t av;
#pragma unroll
                    for (int k = 0; k < 8; k++) av[k] = a[j][m].v[k];
#pragma unroll
                    for (int q = 0; q < NB; q++)
#pragma unroll
                        for (int r = 0; r < kRows; r++) acc[q][m][r] = dot8(av, b[j][q][r], acc[q][m][r]);
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < NB; q++)
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int r = 0; r < kRows; r++) {
                const float v = wave_sum(acc[q][m][r]);
                if (lane == 0) part[wid][(q * M + m) * kRows + r] = v;
            }
    __syncthreads();
    if (EPI == E_QKV) {
        // rotate (queries, keys) and add to the caches (keys, values) with the rounding points of
        // the separate thunks: y = f16(f16(x cos) + f16(rot(x) sin)), cache = f16(cache + y)
        const int m = tid / kRows, r = tid % kRows;
        if (tid < M * kRows) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < W; w++) v += part[w][m * kRows + r];
            float y = rnd16(p.alpha * v);
            if (blockIdx.y < 2) {
                static_assert(kRows == 4, "a column's partner is lane ^ 2");
                const float xp = dpp<0x4E>(y);
                y = rnd16(rnd16(y * h2f(ecos)) + rnd16((r < kRows / 2 ? -xp : xp) * h2f(esin)));
            }
            if (blockIdx.y == 0) {
                p.C[m * p.ldc + ecol] = f2h(y);
            } else {
                (blockIdx.y == 1 ? p.kc : p.vc)[m * p.ldc + ecol] = f2h(h2f(ecell) + y);
            }
        }
        return;
    }
    if (tid < M * kRows) {
        const int m = tid / kRows, r = tid % kRows;
        float v[NB];
#pragma unroll
        for (int q = 0; q < NB; q++) {
            v[q] = 0.f;
#pragma unroll
            for (int w = 0; w < W; w++) v[q] += part[w][(q * M + m) * kRows + r];
        }
        if (EPI == E_PLAIN && p.cand) {
            uint32_t k = n0 + r < p.N ? arg_key(f2h(p.alpha * v[0]), n0 + r) : 0u;
            k = max(k, dpp<0xB1>(k));
            k = max(k, dpp<0x4E>(k));
            if (r == 0) p.cand[(int64_t)m * gridDim.x + blockIdx.x] = k;
        }
        if (n0 + r < p.N) {
            if (GATE) {
                // g = f16(alpha dot_g), u = f16(alpha dot_u); h = f16(f16(silu g) * u)
                const float g = rnd16(p.alpha * v[0]), u = rnd16(p.alpha * v[NB - 1]);
                const float y = rnd16(g / (1.0f + expf(-g)));
                p.C[m * p.ldc + n0 + r] = f2h(y * u);
            } else {
                p.C[m * p.ldc + n0 + r] = f2h(p.alpha * v[0]);
            }
        }
    }
}

// The arg max of each row from the workgroups' candidates, in out_tok; the last row's token is added to in_tok[pos]
// (pos < 0: nowhere), src/librarium/llama.rs:953-959.  One workgroup and a chain of latencies.  (A lane's candidates
// requested together, eight of a vocabulary of 32000: no difference, 4.42 and 4.44 us behind 3 layers of 3200, 4.13 and 4.04 behind
// 4 of 2048 where traces of one kernel differ by 0.2.)
__global__ void __launch_bounds__(1024)
finish_rows_kernel(int M, int count, const uint32_t *__restrict__ cand, uint16_t *out_tok, uint16_t *in_tok, int64_t pos)
{
    __shared__ uint32_t best[16];
    // (read up front: behind the arg max it would be one more round trip to memory)
    const uint16_t before = threadIdx.x == 0 && pos >= 0 ? in_tok[pos] : 0;
    for (int m = 0; m < M; m++) {
        uint32_t k = 0;
        for (int i = threadIdx.x; i < count; i += 1024) k = max(k, cand[(int64_t)m * count + i]);
        k = wave_reduce(k, [](uint32_t a, uint32_t b) { return max(a, b); });
        __syncthreads();
        if ((threadIdx.x & 63) == 0) best[threadIdx.x >> 6] = k;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < 16; w++) k = max(k, best[w]);
            const uint16_t id = k ? (uint16_t)(0xffff - (k & 0xffff)) : 0;     // (a row of NaNs alone has no candidate)
            out_tok[m] = id;
            if (m == M - 1 && pos >= 0) in_tok[pos] = (uint16_t)(before + id);
        }
    }
}

template <int M, bool NORM, int EPI, int W, int kPre>
void launch_cfg(const SkinnyArgs &p, hipStream_t st)
{
    const dim3 grid((unsigned)((p.N + kRows - 1) / kRows), EPI == E_QKV ? 3 : 1), block(W * 64);
    hipLaunchKernelGGL((gemm_skinny_nt_kernel<M, NORM, EPI, W, kPre>), grid, block, 0, st, p);
}

// How a row of K is cut over lanes.  Lanes without a piece of their own still load (a duplicate), so one row takes as many
// pieces per lane as it needs: K = 2048 is one piece per lane of 4 waves (with two: gate and up 11.5 against 10.3 us, a
// head of 32000 25.5 against 22.0), and up to 1024 one wave does, so that no barrier stands between its loads and its
// result.  A plain product of 8200 to 10240 elements is five pieces in one pass (K = 8640: four in two passes 13.2
// against 11.5); every longer row is passes of four, the last of them partly duplicates, and two to four rows have
// passes of two (K <= 4096) or four pieces only: no other cut of those has been measured.  Eight columns per
// workgroup instead of four changed nothing (13.9 and 14.1 us for q, k, v of 3200).
template <bool NORM, int EPI>
int launch(int64_t M, const SkinnyArgs &p, hipStream_t st)
{
    const int64_t pieces = p.K / 8;
    if (M == 1) {
        if (pieces <= 64) launch_cfg<1, NORM, EPI, 1, 1>(p, st);
        else if (pieces <= 128) launch_cfg<1, NORM, EPI, 1, 2>(p, st);
        else if (pieces <= 256) launch_cfg<1, NORM, EPI, 4, 1>(p, st);
        else if (pieces <= 512) launch_cfg<1, NORM, EPI, 4, 2>(p, st);
        else if (pieces <= 768) launch_cfg<1, NORM, EPI, 4, 3>(p, st);
        else if (!NORM && EPI == E_PLAIN && pieces > 1024 && pieces <= 1280) launch_cfg<1, false, E_PLAIN, 4, 5>(p, st);
        else launch_cfg<1, NORM, EPI, 4, 4>(p, st);
    } else if (pieces <= 512) {
        if (M == 2) launch_cfg<2, NORM, EPI, 4, 2>(p, st);
        else if (M == 3) launch_cfg<3, NORM, EPI, 4, 2>(p, st);
        else launch_cfg<4, NORM, EPI, 4, 2>(p, st);
    } else {
        if (M == 2) launch_cfg<2, NORM, EPI, 4, 4>(p, st);
        else if (M == 3) launch_cfg<3, NORM, EPI, 4, 4>(p, st);
        else launch_cfg<4, NORM, EPI, 4, 4>(p, st);
    }
    return launch_status("gemm_skinny_nt");
}

}  // namespace

// A, B rows 16-byte aligned (lda, ldb multiples of 8), K % 8 == 0, 1 <= M <= 4
int gemm_skinny_nt_launch(int64_t M, int64_t N, int64_t K, float alpha, const half_t *A, int64_t lda,
                          const half_t *B, int64_t ldb, half_t *C, int64_t ldc, hipStream_t st)
{
    SkinnyArgs p = {};
    p.N = N; p.K = K; p.alpha = alpha;
    p.A = A; p.lda = lda;
    p.B = B; p.ldb = ldb;
    p.C = C; p.ldc = ldc;
    return launch<false, E_PLAIN>(M, p, st);
}

namespace {

SkinnyArgs norm_args(const RowSource &x, int64_t N, int64_t K, void *sum_out)
{
    SkinnyArgs p = {};
    p.N = N; p.K = K; p.alpha = 1.0f;
    p.A = (const half_t *)x.x; p.lda = K;
    p.x2 = (const half_t *)x.x2;
    p.w = (const half_t *)x.w_norm; p.eps = x.eps;
    p.tok = x.tok; p.vocab = x.vocab; p.status = x.status;
    p.sum_out = (half_t *)sum_out;
    p.ldb = K;
    p.ldc = N;
    return p;
}

}  // namespace

int rows_qkv_launch(int64_t M, int64_t H, int64_t Dh, const RowSource &x, void *sum_out, const void *Wq, const void *Wk, const void *Wv,
                    const void *cos16, const void *sin16, void *q_rot, void *k_cache_rows, void *v_cache_rows, hipStream_t st)
{
    const int64_t D = H * Dh;
    SkinnyArgs p = norm_args(x, D, D, sum_out);
    p.B = (const half_t *)Wq; p.B2 = (const half_t *)Wk; p.B3 = (const half_t *)Wv;
    p.C = (half_t *)q_rot;
    p.cos16 = (const half_t *)cos16; p.sin16 = (const half_t *)sin16;
    p.kc = (half_t *)k_cache_rows; p.vc = (half_t *)v_cache_rows;
    p.H = (int)H; p.Dh = (int)Dh;
    p.half_head.set((uint32_t)(Dh / 2));
    return launch<true, E_QKV>(M, p, st);
}

int rows_gate_launch(int64_t M, int64_t N, int64_t K, const RowSource &x, void *sum_out, const void *B, const void *B_mul, void *C,
                     hipStream_t st)
{
    SkinnyArgs p = norm_args(x, N, K, sum_out);
    p.B = (const half_t *)B; p.B2 = (const half_t *)B_mul;
    p.C = (half_t *)C;
    return launch<true, E_GATE>(M, p, st);
}

int rows_norm_launch(int64_t M, int64_t N, int64_t K, const RowSource &x, const void *B, void *C, hipStream_t st)
{
    SkinnyArgs p = norm_args(x, N, K, nullptr);
    p.B = (const half_t *)B;
    p.C = (half_t *)C;
    return launch<true, E_PLAIN>(M, p, st);
}

size_t rows_head_scratch_bytes(int64_t M, int64_t N) { return (size_t)M * (size_t)((N + kRows - 1) / kRows) * sizeof(uint32_t); }

int rows_head_launch(int64_t M, int64_t N, int64_t K, const RowSource &x, const void *B, void *logit, void *scratch, void *out_tok,
                     void *in_tok, int64_t pos, hipStream_t st)
{
    CACTI_REQUIRE(N <= 65536, CACTI_E_NOTIMPL, "rows_head: more than 65536 tokens");
    SkinnyArgs p = norm_args(x, N, K, nullptr);
    p.B = (const half_t *)B;
    p.C = (half_t *)logit;
    p.cand = (uint32_t *)scratch;
    const int rc = launch<true, E_PLAIN>(M, p, st);
    if (rc) return rc;
    hipLaunchKernelGGL(finish_rows_kernel, dim3(1), dim3(1024), 0, st, (int)M, (int)((N + kRows - 1) / kRows), (const uint32_t *)scratch,
                       (uint16_t *)out_tok, (uint16_t *)in_tok, pos);
    return launch_status("finish_rows");
}

}  // namespace cacti

using namespace cacti;

CACTI_API int cacti_hip_rows_norm_matmul_f16(int64_t M, int64_t N, int64_t K, const void *x, const void *x2,
                                             const void *w_norm, float eps, void *sum_out, const void *B,
                                             const void *B_mul, void *C, void *stream)
{
    CACTI_REQUIRE(M >= 1 && M <= 4, CACTI_E_NOTIMPL, "rows_norm_matmul: 1 to 4 rows are handled here (M=%lld)", (long long)M);
    CACTI_REQUIRE(N > 0 && K > 0 && K % 8 == 0 && K <= 8 * kMaxNorm, CACTI_E_NOTIMPL,
                  "rows_norm_matmul: need K %% 8 == 0 and K <= %d (K=%lld)", 8 * kMaxNorm, (long long)K);
    CACTI_REQUIRE(x && B && C && (w_norm || (!x2 && !sum_out)), CACTI_E_INVALID, "rows_norm_matmul: null pointer");
    CACTI_REQUIRE(aligned(x, 16) && aligned(x2, 16) && aligned(w_norm, 16) && aligned(sum_out, 16) && aligned(B, 16) &&
                      aligned(B_mul, 16) && aligned(C, 2),
                  CACTI_E_INVALID, "rows_norm_matmul: operands must be 16-byte aligned");
    SkinnyArgs p = norm_args(RowSource{x, x2, w_norm, eps, nullptr, 0, nullptr}, N, K, sum_out);
    p.B = (const half_t *)B; p.B2 = (const half_t *)B_mul;
    p.C = (half_t *)C;
    hipStream_t st = (hipStream_t)stream;
    if (w_norm) return B_mul ? launch<true, E_GATE>(M, p, st) : launch<true, E_PLAIN>(M, p, st);
    return B_mul ? launch<false, E_GATE>(M, p, st) : launch<false, E_PLAIN>(M, p, st);
}

CACTI_API int cacti_hip_rows_qkv_rope_cache_f16(int64_t M, int64_t H, int64_t Dh, const void *x, const void *x2,
                                                const void *w_norm, float eps, void *sum_out, const void *Wq,
                                                const void *Wk, const void *Wv, const void *cos16, const void *sin16,
                                                void *q_rot, void *k_cache_rows, void *v_cache_rows, void *stream)
{
    const int64_t D = H * Dh;
    CACTI_REQUIRE(M >= 1 && M <= 4, CACTI_E_NOTIMPL, "rows_qkv: 1 to 4 rows are handled here (M=%lld)", (long long)M);
    CACTI_REQUIRE(H > 0 && Dh > 0 && Dh % 4 == 0 && D % 8 == 0 && D <= 8 * kMaxNorm, CACTI_E_NOTIMPL,
                  "rows_qkv: need Dh %% 4 == 0, H*Dh %% 8 == 0 and H*Dh <= %d", 8 * kMaxNorm);
    CACTI_REQUIRE(x && w_norm && Wq && Wk && Wv && cos16 && sin16 && q_rot && k_cache_rows && v_cache_rows, CACTI_E_INVALID,
                  "rows_qkv: null pointer");
    CACTI_REQUIRE(aligned(x, 16) && aligned(x2, 16) && aligned(w_norm, 16) && aligned(sum_out, 16) && aligned(Wq, 16) &&
                      aligned(Wk, 16) && aligned(Wv, 16) && aligned(cos16, 2) && aligned(sin16, 2) && aligned(q_rot, 2) &&
                      aligned(k_cache_rows, 2) && aligned(v_cache_rows, 2),
                  CACTI_E_INVALID, "rows_qkv: rows and weights must be 16-byte aligned");
    return rows_qkv_launch(M, H, Dh, RowSource{x, x2, w_norm, eps, nullptr, 0, nullptr}, sum_out, Wq, Wk, Wv, cos16, sin16, q_rot,
                           k_cache_rows, v_cache_rows, (hipStream_t)stream);
}
