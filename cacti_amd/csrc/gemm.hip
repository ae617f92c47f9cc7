// f16 x f16 -> fp32-accumulate -> f16 GEMM on gfx950 MFMA (v_mfma_f32_32x32x16_f16),
// C = alpha op(A) op(B) + beta C, row-major, all four transpose cases, optional
// strided batch (the per-head blocks of attention tensors).
//
// Block tile BM x BN x BK, 256 lanes = 4 wavefronts in a 2 x 2 grid, each wavefront
// owning a (BM/2) x (BN/2) tile of 32 x 32 MFMA accumulators.  Both operands are staged
// in LDS as [row][k] with k contiguous (row = m for A, n for B) and a padded row stride
// so that the 16-byte operand reads of a wavefront hit distinct banks.  An operand whose
// k index is not contiguous in memory (A^T, or B not transposed) is transposed in
// registers on its way from global memory to LDS, so the MFMA read path is the same for
// all four cases.  Global loads for tile t+1 are issued before the MFMAs of tile t and
// land in the other LDS buffer afterwards: one barrier per k tile.
//
// The MFMA is issued with the B fragment as first operand, so a lane ends up with 4
// consecutive columns of one row of C per accumulator group and stores 8 bytes at a time.
#include <stdlib.h>

#include "common.h"
#include "gemm_internal.h"

using namespace cacti;

namespace {

template <int VEC> struct VecT;
template <> struct VecT<8> { typedef uint4 type; };
template <> struct VecT<4> { typedef uint2 type; };
template <> struct VecT<1> { typedef uint16_t type; };

template <int VEC>
__device__ __forceinline__ typename VecT<VEC>::type vzero();
template <> __device__ __forceinline__ uint4 vzero<8>() { return make_uint4(0, 0, 0, 0); }
template <> __device__ __forceinline__ uint2 vzero<4>() { return make_uint2(0, 0); }
template <> __device__ __forceinline__ uint16_t vzero<1>() { return 0; }

template <int VEC>
__device__ __forceinline__ uint16_t vget(const typename VecT<VEC>::type &v, int j)
{
    return reinterpret_cast<const uint16_t *>(&v)[j];
}

constexpr int BM = 128, BN = 128, BK = 32, PAD = 8, LDS_LD = BK + PAD, NT = 256;

// ---- global -> registers ----------------------------------------------------
// K-contiguous operand: tile [ROWS][BK], vectors of VEC halves along k.
template <int ROWS, int VEC>
struct LoadKC {
    static constexpr int CPR = BK / VEC;                  // chunks per row
    static constexpr int ITEMS = ROWS * CPR;
    static constexpr int NL = (ITEMS + NT - 1) / NT;
    typename VecT<VEC>::type st[NL];

    __device__ __forceinline__ void load(const half_t *base, int64_t ld, int64_t row0, int64_t R,
                                         int64_t k0, int64_t K)
    {
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT;
            const int row = c / CPR, kc = c % CPR;
            const int64_t gr = row0 + row, gk = k0 + kc * VEC;
            if (c < ITEMS && gr < R && gk < K)
                st[it] = *reinterpret_cast<const typename VecT<VEC>::type *>(base + gr * ld + gk);
            else
                st[it] = vzero<VEC>();
        }
    }
    __device__ __forceinline__ void store(half_t *lds)
    {
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT;
            const int row = c / CPR, kc = c % CPR;
            if (c < ITEMS)
                *reinterpret_cast<typename VecT<VEC>::type *>(lds + row * LDS_LD + kc * VEC) =
                    st[it];
        }
    }
};

// K-strided operand: memory is [k][row]; blocks of 4 k x VEC rows, transposed in registers.
template <int ROWS, int VEC>
struct LoadKS {
    static constexpr int RC = ROWS / VEC;                 // row chunks
    static constexpr int ITEMS = (BK / 4) * RC;
    static constexpr int NL = (ITEMS + NT - 1) / NT;
    typename VecT<VEC>::type st[NL][4];

    __device__ __forceinline__ void load(const half_t *base, int64_t ld, int64_t row0, int64_t R,
                                         int64_t k0, int64_t K)
    {
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT;
            const int rc = c % RC, kq = c / RC;
            const int64_t gr = row0 + rc * VEC;
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                const int64_t gk = k0 + kq * 4 + kk;
                if (c < ITEMS && gr < R && gk < K)
                    st[it][kk] =
                        *reinterpret_cast<const typename VecT<VEC>::type *>(base + gk * ld + gr);
                else
                    st[it][kk] = vzero<VEC>();
            }
        }
    }
    __device__ __forceinline__ void store(half_t *lds)
    {
#pragma unroll
        for (int it = 0; it < NL; it++) {
            const int c = threadIdx.x + it * NT;
            const int rc = c % RC, kq = c / RC;
            if (c < ITEMS) {
#pragma unroll
                for (int j = 0; j < VEC; j++) {
                    uint2 w;
                    w.x = (uint32_t)vget<VEC>(st[it][0], j) | ((uint32_t)vget<VEC>(st[it][1], j) << 16);
                    w.y = (uint32_t)vget<VEC>(st[it][2], j) | ((uint32_t)vget<VEC>(st[it][3], j) << 16);
                    *reinterpret_cast<uint2 *>(lds + (rc * VEC + j) * LDS_LD + kq * 4) = w;
                }
            }
        }
    }
};

template <bool KSTRIDED, int ROWS, int VEC> struct Loader;
template <int ROWS, int VEC> struct Loader<false, ROWS, VEC> : LoadKC<ROWS, VEC> {};
template <int ROWS, int VEC> struct Loader<true, ROWS, VEC> : LoadKS<ROWS, VEC> {};

template <bool TA, bool TB, int VEC>
__global__ void __launch_bounds__(NT) gemm_f16_kernel(GemmArgs p)
{
    __shared__ __attribute__((aligned(16))) half_t As[2][BM * LDS_LD];
    __shared__ __attribute__((aligned(16))) half_t Bs[2][BN * LDS_LD];

    const int tile = blockIdx.x;
    const int tm = tile % p.tiles_m, tn = tile / p.tiles_m;
    const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
    const int64_t bz = blockIdx.z;
    const half_t *A = p.A + bz * p.sa;
    const half_t *B = p.B + bz * p.sb;
    half_t *C = p.C + bz * p.sc;

    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int wm = wid & 1, wn = wid >> 1;
    const int l32 = lane & 31, lh = lane >> 5;

    // A is k-strided in memory when transposed; B when not transposed
    Loader<TA, BM, VEC> la;
    Loader<!TB, BN, VEC> lb;

    float16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    int nk = (int)((p.K + BK - 1) / BK), kt0 = 0;
    if (p.tri == 1 && n0 > m0 + BM - 1) return;               // uniform for the block
    if (p.tri == 2) nk = min(nk, (int)((m0 + BM + BK - 1) / BK));
    if (p.tri == 3) kt0 = (int)(m0 / BK);
    la.load(A, p.lda, m0, p.M, (int64_t)kt0 * BK, p.K);
    lb.load(B, p.ldb, n0, p.N, (int64_t)kt0 * BK, p.K);
    la.store(As[kt0 & 1]);
    lb.store(Bs[kt0 & 1]);
    __syncthreads();

    for (int kt = kt0; kt < nk; kt++) {
        const int cur = kt & 1;
        if (kt + 1 < nk) {
            la.load(A, p.lda, m0, p.M, (int64_t)(kt + 1) * BK, p.K);
            lb.load(B, p.ldb, n0, p.N, (int64_t)(kt + 1) * BK, p.K);
        }
        const half_t *as = As[cur] + (wm * 64 + l32) * LDS_LD + lh * 8;
        const half_t *bs = Bs[cur] + (wn * 64 + l32) * LDS_LD + lh * 8;
#pragma unroll
        for (int ks = 0; ks < BK / 16; ks++) {
            half8_t af[2], bf[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                af[i] = *reinterpret_cast<const half8_t *>(as + i * 32 * LDS_LD + ks * 16);
                bf[i] = *reinterpret_cast<const half8_t *>(bs + i * 32 * LDS_LD + ks * 16);
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] =
                        __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[j], af[i], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) {
            la.store(As[cur ^ 1]);
            lb.store(Bs[cur ^ 1]);
        }
        __syncthreads();
    }

    // epilogue: lane holds row m = .. + l32 and, per accumulator group q, the 4
    // consecutive columns n = .. + 8 q + 4 lh + {0..3}
    const bool has_beta = p.beta != 0.f;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int64_t m = m0 + wm * 64 + i * 32 + l32;
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int64_t n = n0 + wn * 64 + j * 32 + q * 8 + lh * 4;
                half_t *cp = C + m * p.ldc + n;
                if (VEC >= 4) {
                    if (n < p.N) {
                        half4_t o;
                        if (has_beta) {
                            half4_t old = *reinterpret_cast<const half4_t *>(cp);
#pragma unroll
                            for (int r = 0; r < 4; r++)
                                o[r] = f2h(p.alpha * acc[i][j][q * 4 + r] + p.beta * h2f(old[r]));
                        } else {
#pragma unroll
                            for (int r = 0; r < 4; r++) o[r] = f2h(p.alpha * acc[i][j][q * 4 + r]);
                        }
                        *reinterpret_cast<half4_t *>(cp) = o;
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        if (n + r < p.N) {
                            float v = p.alpha * acc[i][j][q * 4 + r];
                            if (has_beta) v += p.beta * h2f(cp[r]);
                            cp[r] = f2h(v);
                        }
                    }
                }
            }
        }
    }
}

template <bool TA, bool TB>
int launch_vec(int vec, const GemmArgs &p, int64_t nblk, hipStream_t st)
{
    dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, (unsigned)nblk), block(NT);
    if (vec == 8)
        hipLaunchKernelGGL((gemm_f16_kernel<TA, TB, 8>), grid, block, 0, st, p);
    else if (vec == 4)
        hipLaunchKernelGGL((gemm_f16_kernel<TA, TB, 4>), grid, block, 0, st, p);
    else
        hipLaunchKernelGGL((gemm_f16_kernel<TA, TB, 1>), grid, block, 0, st, p);
    return launch_status("gemm_f16");
}

inline bool mult(int64_t v, int64_t a) { return v % a == 0; }

// The tile kernels keep a lane's place inside a tile (up to 256 rows) as a 32-bit byte offset; operands whose rows lie
// farther apart go to the kernel above, which addresses each element in 64 bits.
constexpr int64_t kMaxPitch = (int64_t)1 << 23;

}  // namespace

namespace {

// ws_need null: the caller has no workspace.  Otherwise *ws_need is set to the bytes the chosen way needs (of those that need no
// more than `most`), and if that is more than ws_bytes nothing is launched.
int gemm_run(int ta, int tb, int64_t nblk, int64_t M, int64_t N, int64_t K, float alpha, const void *A, int64_t lda,
             int64_t stride_a, const void *B, int64_t ldb, int64_t stride_b, float beta, void *C, int64_t ldc,
             int64_t stride_c, int tri, size_t most, void *ws, size_t ws_bytes, size_t *ws_need, void *stream)
{
    CACTI_REQUIRE(tri >= 0 && tri <= 3, CACTI_E_INVALID, "gemm: tri must be 0..3");
    CACTI_REQUIRE(tri == 0 || (tri == 1 && M == N) || (tri == 2 && !ta && M == K) ||
                      (tri == 3 && ta && M == K),
                  CACTI_E_INVALID, "gemm: tri=%d needs a square (sequence x sequence) operand", tri);
    CACTI_REQUIRE(A && B && C, CACTI_E_INVALID, "gemm: null operand");
    CACTI_REQUIRE(M > 0 && N > 0 && K > 0 && nblk > 0 && nblk <= 65535, CACTI_E_INVALID,
                  "gemm: bad shape M=%lld N=%lld K=%lld nblk=%lld", (long long)M, (long long)N,
                  (long long)K, (long long)nblk);
    CACTI_REQUIRE(beta == 0.f || beta == 1.f, CACTI_E_INVALID, "gemm: beta must be 0 or 1");
    CACTI_REQUIRE(lda >= (ta ? M : K) && ldb >= (tb ? K : N) && ldc >= N, CACTI_E_INVALID,
                  "gemm: leading dimension smaller than the row length");
    CACTI_REQUIRE(aligned(A, 2) && aligned(B, 2) && aligned(C, 2), CACTI_E_INVALID,
                  "gemm: operands must be 2-byte aligned");
    CACTI_REQUIRE(!ws_need || aligned(ws, 16), CACTI_E_INVALID, "gemm: the workspace must be 16-byte aligned");
    GemmArgs p = {};
    p.M = M; p.N = N; p.K = K; p.alpha = alpha; p.beta = beta;
    p.A = (const half_t *)A; p.lda = lda; p.sa = stride_a;
    p.B = (const half_t *)B; p.ldb = ldb; p.sb = stride_b;
    p.C = (half_t *)C; p.ldc = ldc; p.sc = stride_c;
    p.tiles_m = (int)((M + BM - 1) / BM);
    p.tiles_n = (int)((N + BN - 1) / BN);
    p.tri = tri;
    CACTI_REQUIRE((int64_t)p.tiles_m * p.tiles_n < (1LL << 31), CACTI_E_NOTIMPL, "gemm: too many tiles");
    if (ws_need) *ws_need = 0;

    // widest vector every operand supports: contiguous extent, leading dimension,
    // batch stride and base address must all be multiples of it
    const int64_t ca = ta ? M : K, cb = tb ? K : N;
    const bool multi = nblk > 1;
    auto fits_a = [&](int v) { return mult(ca, v) && mult(lda, v) && (!multi || mult(stride_a, v)) && aligned(A, 2 * v); };
    auto fits_b = [&](int v) { return mult(cb, v) && mult(ldb, v) && (!multi || mult(stride_b, v)) && aligned(B, 2 * v); };
    auto fits_c = [&](int v) { return mult(N, v) && mult(ldc, v) && (!multi || mult(stride_c, v)) && aligned(C, 2 * v); };
    int vec = 1;
    for (int v : {8, 4})
        if (fits_a(v) && fits_b(v) && fits_c(v)) {
            vec = v;
            break;
        }
    hipStream_t st = (hipStream_t)stream;
    const bool near = lda < kMaxPitch && ldb < kMaxPitch;
    // Scores: a batch of heads, or the lower triangle of one.  (A single product with a short K is no score: 149 x 8280 x 96
    // takes 43 us there, whose workgroups walk tile rows of a square, and 4.3 on the tiles below; 2048 x 2048 x 128 17 and 5.9.)
    if (vec >= 4 && !ta && tb && K <= 128 && beta == 0.f && tri <= 1 && (nblk > 1 || tri == 1 || (vec < 8 && !ws_need)))
        return gemm_nt_smallk_launch(p, nblk, st);
    // one to four rows against a weight matrix (decoding): a stream over B
    if (vec == 8 && !ta && tb && M <= 4 && nblk == 1 && beta == 0.f && tri == 0)
        return gemm_skinny_nt_launch(M, N, K, alpha, p.A, lda, p.B, ldb, p.C, ldc, st);
    // The attention products with a [sequence, heads, head_dim] operand: A (probabilities or
    // their adjoint) is 16-byte aligned, B and C are per-head slabs whose offset (head_dim 100)
    // is only a multiple of 8 bytes.  Addressed from the 16-byte boundary below each slab they
    // take the direct-load path; the extra columns read stay inside the columns the blocks
    // cover in one row of B (checked here).
    if (near && vec == 4 && !tb && nblk > 1 && mult(K, 64) && mult(ta ? M : K, 8) && mult(lda, 8) &&
        mult(stride_a, 8) && aligned(A, 16) && mult(ldb, 8) && mult(ldc, 8) && aligned(B, 16) &&
        aligned(C, 16) && (stride_b & 7) == (stride_c & 7)) {
        const int64_t row_end = (nblk - 1) * stride_b + N;
        bool inside = stride_b >= 0 && row_end <= ldb;
        for (int64_t bz = 0; bz < nblk && inside; bz++) {
            const int64_t shift = (bz * stride_b) & 7;
            const int64_t first = bz * stride_b - shift;          // >= 0: bz * stride_b >= shift
            inside = first + (shift + N + 7) / 8 * 8 <= row_end;
        }
        if (inside) {
            p.win = 1;
            return gemm_mfma_launch(ta, tb, p, nblk, 8, st);
        }
    }
    if (near && tri == 0 && vec == 8) {
        const GemmPlan plan = gemm_plan(M, N, K, nblk, ws_need ? most : 0);
        if (plan.split > 1) {
            p.ldp = gemm_part_pitch(N);
            p.part = (float *)ws;
            *ws_need = gemm_parts_bytes(M, N, plan.split);
            if (*ws_need > ws_bytes) return 0;
        }
        return gemm_direct_launch(ta, tb, p, nblk, plan, st);
    }
    // Operands that are not 16-byte aligned, with a workspace: loaded as they are through registers on 64 x 64 tiles, or laid
    // out anew for the direct kernels (one launch for both, some 3.5 us and 0.4 us per MB), whichever is expected to take
    // less.  Over 85 products of M 9 .. 4000, N 50 .. 5000, K 66 .. 5000 in three layouts the copy takes 28 % longer in the
    // mean than the better of the two, registers 3 %, this rule 0.2 % (19 % at worst: 687 x 3731 x 410).  Element-wise loads
    // in the kernel cost 1.6 us (both operands contiguous in K) to 3.4 us (both strided) per 32 values of K instead.
    const int64_t ra = ta ? K : M, rb = tb ? N : K, pa = (ca + 7) / 8 * 8, pb = (cb + 7) / 8 * 8;
    const bool ok_a = fits_a(8) && lda < kMaxPitch, ok_b = fits_b(8) && ldb < kMaxPitch, as_it_is = near && ca >= 8 && cb >= 8;
    size_t bytes_a = ok_a ? 0 : (size_t)ra * (size_t)pa * 2, bytes_b = ok_b ? 0 : (size_t)rb * (size_t)pb * 2;
    const bool copied = bytes_a + bytes_b <= most;
    if (ws_need && tri == 0 && nblk == 1 && K >= 8 && pa < kMaxPitch && pb < kMaxPitch && (copied || as_it_is)) {
        GemmPlan plan = gemm_plan(M, N, K, 1, copied ? most - (bytes_a + bytes_b) : 0);
        if (as_it_is) {
            const GemmPlan as_is = gemm_plan_any(M, N, K, most);
            const double copy = bytes_a + bytes_b > 0 ? 3.5 + (double)(bytes_a + bytes_b) / 2.5e6 : 0;
            if (!copied || as_is.us < plan.us + copy) {
                plan = as_is;
                p.any = 1;
                bytes_a = bytes_b = 0;
            }
        }
        p.ldp = gemm_part_pitch(N);
        const size_t bytes_part = plan.split > 1 ? gemm_parts_bytes(M, N, plan.split) : 0;
        *ws_need = bytes_a + bytes_b + bytes_part;                // each a multiple of 16
        if (*ws_need > ws_bytes) return 0;
        char *w = static_cast<char *>(ws);
        const half_t *src[2] = {p.A, p.B};
        half_t *dst[2] = {bytes_a ? (half_t *)w : nullptr, bytes_b ? (half_t *)(w + bytes_a) : nullptr};
        const int64_t rows[2] = {ra, rb}, cols[2] = {ca, cb}, ld[2] = {lda, ldb};
        if (bytes_a + bytes_b > 0) {
            const int rc = gemm_repack(src, dst, rows, cols, ld, st);
            if (rc) return rc;
        }
        if (bytes_a) {
            p.A = dst[0];
            p.lda = pa;
        }
        if (bytes_b) {
            p.B = dst[1];
            p.ldb = pb;
        }
        p.part = (float *)(w + bytes_a + bytes_b);
        p.odd = !fits_c(8);
        return gemm_direct_launch(ta, tb, p, 1, plan, st);
    }
    if (near && vec >= 4) return gemm_mfma_launch(ta, tb, p, nblk, vec, st);
    if (!ta && !tb) return launch_vec<false, false>(vec, p, nblk, st);
    if (!ta && tb) return launch_vec<false, true>(vec, p, nblk, st);
    if (ta && !tb) return launch_vec<true, false>(vec, p, nblk, st);
    return launch_vec<true, true>(vec, p, nblk, st);
}

}  // namespace

CACTI_API int cacti_hip_gemm_f16_strided_batched_tri(int ta, int tb, int64_t nblk, int64_t M,
                                                     int64_t N, int64_t K, float alpha, const void *A,
                                                     int64_t lda, int64_t stride_a, const void *B,
                                                     int64_t ldb, int64_t stride_b, float beta,
                                                     void *C, int64_t ldc, int64_t stride_c, int tri,
                                                     void *stream)
{
    return gemm_run(ta, tb, nblk, M, N, K, alpha, A, lda, stride_a, B, ldb, stride_b, beta, C, ldc, stride_c, tri, 0, nullptr, 0,
                    nullptr, stream);
}

namespace cacti {
int gemm_f16_within(size_t most, int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha, const void *A, int64_t lda, const void *B, int64_t ldb,
                    float beta, void *C, int64_t ldc, void *ws, size_t ws_bytes, size_t *ws_need, hipStream_t st)
{
    return gemm_run(ta, tb, 1, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 0, most, ws, ws_bytes, ws_need, st);
}

int gemm_parts_within(size_t most, int ta, int tb, int64_t M, int64_t N, int64_t K, bool acc)
{
    if (!mult(N, 8) || !mult(ta ? M : K, 8) || !mult(tb ? K : N, 8) || (ta ? M : K) >= kMaxPitch || (tb ? K : N) >= kMaxPitch) return 1;
    if (!ta && tb && M <= 4 && !acc) return 1;                    // a stream over B
    return gemm_plan(M, N, K, 1, most).split;
}
}  // namespace cacti

CACTI_API int cacti_hip_gemm_f16_ws(int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha, const void *A, int64_t lda,
                                    const void *B, int64_t ldb, float beta, void *C, int64_t ldc, void *ws, size_t ws_bytes,
                                    size_t *ws_need, void *stream)
{
    CACTI_REQUIRE(ws_need, CACTI_E_INVALID, "gemm_ws: null ws_need");
    return gemm_f16_within(SIZE_MAX, ta, tb, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, ws, ws_bytes, ws_need, (hipStream_t)stream);
}

CACTI_API int cacti_hip_gemm_plan(int64_t M, int64_t N, int64_t K, int64_t nz, int64_t out[6])
{
    CACTI_REQUIRE(out && M > 0 && N > 0 && K > 0 && nz > 0, CACTI_E_INVALID, "gemm_plan: bad argument");
    const GemmPlan plan = gemm_plan(M, N, K, nz, 0);
    gemm_tile_dims(plan.tile, out, out + 1);
    out[2] = plan.cols > 0 ? plan.cols : N;
    gemm_tile_dims(plan.rest, out + 3, out + 4);
    out[5] = plan.cols > 0 ? 2 : 1;
    return 0;
}

CACTI_API int cacti_hip_gemm_plan_ws(int64_t M, int64_t N, int64_t K, size_t lent, int parts, int64_t out[3], double *us)
{
    CACTI_REQUIRE(out && us && M > 0 && N > 0 && K > 0 && parts >= 0 && parts <= 8, CACTI_E_INVALID, "gemm_plan_ws: bad argument");
    const GemmPlan plan = parts > 1 ? gemm_plan_parts(M, N, K, parts) : gemm_plan(M, N, K, 1, parts == 0 ? lent : 0);
    out[0] = plan.tile < 0 ? 0 : plan.split;
    gemm_tile_dims(plan.tile < 0 ? 0 : plan.tile, out + 1, out + 2);
    *us = plan.us;
    return 0;
}

CACTI_API int cacti_hip_gemm_kernel_name(int ta, int tb, int64_t M, int64_t N, int64_t K, int64_t nz, char *name, size_t bytes)
{
    CACTI_REQUIRE(name && M > 0 && N > 0 && K > 0 && nz > 0, CACTI_E_INVALID, "gemm_kernel_name: bad argument");
    const int n = gemm_kernel_name(ta, tb, gemm_plan(M, N, K, nz, 0), name, bytes);
    CACTI_REQUIRE(n >= 0 && (size_t)n < bytes, CACTI_E_INVALID, "gemm_kernel_name: %zu bytes are too few for the name", bytes);
    return 0;
}

// Pointer-array batch (cublasGemmBatchedEx shape): the products must have one shape; up to
// kMaxPtrBatch of them share a launch when every operand is 16-byte aligned, otherwise they run
// one after another.
CACTI_API int cacti_hip_gemm_f16_batched(int ta, int tb, int64_t nblk, int64_t M, int64_t N, int64_t K,
                                         float alpha, const void *const *A, int64_t lda, const void *const *B,
                                         int64_t ldb, float beta, void *const *C, int64_t ldc, void *stream)
{
    CACTI_REQUIRE(nblk > 0 && A && B && C, CACTI_E_INVALID, "gemm_batched: null pointer array or empty batch");
    for (int64_t z = 0; z < nblk; z++)
        CACTI_REQUIRE(A[z] && B[z] && C[z], CACTI_E_INVALID, "gemm_batched: null operand in block %lld", (long long)z);
    const int64_t ca = ta ? M : K, cb = tb ? K : N;
    bool fast = M > 0 && N > 0 && K > 0 && (beta == 0.f || beta == 1.f) && mult(ca, 8) && mult(cb, 8) && mult(N, 8) &&
                mult(lda, 8) && mult(ldb, 8) && mult(ldc, 8) && lda >= ca && ldb >= cb && ldc >= N && K > 128 &&
                lda < kMaxPitch && ldb < kMaxPitch;
    if (!ta && tb && M <= 4 && beta == 0.f) fast = false;         // a stream over B each, as alone (gemm_run)
    for (int64_t z = 0; z < nblk && fast; z++) fast = aligned(A[z], 16) && aligned(B[z], 16) && aligned(C[z], 16);
    for (int64_t z0 = 0; z0 < nblk; z0 += kMaxPtrBatch) {
        const int64_t cnt = nblk - z0 < kMaxPtrBatch ? nblk - z0 : kMaxPtrBatch;
        if (!fast || cnt == 1) {
            for (int64_t z = z0; z < z0 + cnt; z++) {
                const int rc = cacti_hip_gemm_f16(ta, tb, M, N, K, alpha, A[z], lda, B[z], ldb, beta, C[z], ldc, stream);
                if (rc) return rc;
            }
            continue;
        }
        GemmArgs p = {};
        p.M = M; p.N = N; p.K = K; p.alpha = alpha; p.beta = beta;
        p.A = (const half_t *)A[z0]; p.lda = lda; p.sa = 0;
        p.B = (const half_t *)B[z0]; p.ldb = ldb; p.sb = 0;
        p.C = (half_t *)C[z0]; p.ldc = ldc; p.sc = 0;
        p.ztab = 1;
        for (int64_t z = 0; z < kMaxPtrBatch; z++) {
            const int64_t zz = z0 + (z < cnt ? z : 0);
            p.za[z] = (const half_t *)A[zz] - p.A;
            p.zb[z] = (const half_t *)B[zz] - p.B;
            p.zc[z] = (half_t *)C[zz] - p.C;
        }
        const GemmPlan plan = gemm_plan(M, N, K, cnt, 0);
        const int rc = gemm_direct_launch(ta, tb, p, cnt, plan, (hipStream_t)stream);
        if (rc) return rc;
    }
    return 0;
}

// Whether a chain of aligned operands goes as its plan says: where every product is of whole k tiles, and where the plans expect
// less of it than of the launches one by one, which is nearly everywhere: they spend 3.7 to 6 us each on their start and end.
static bool chain_pays(int64_t n, int64_t M, int64_t N, int64_t K, GemmPlan *plan)
{
    if (!(n > 1 && n <= kMaxPtrBatch && M > 0 && N > 0 && K >= 4 * 64 && mult(K, 64) && mult(N, 8))) return false;
    *plan = gemm_plan_chain(M, N, K, (int)n);
    return plan->us < (double)n * gemm_plan(M, N, K, 1, 0).us;
}

CACTI_API int cacti_hip_gemm_chain_kernel_name(int64_t n, int64_t M, int64_t N, int64_t K, char *name, size_t bytes, int *launches)
{
    CACTI_REQUIRE(name && bytes && launches && n > 0 && M > 0 && N > 0 && K > 0, CACTI_E_INVALID, "gemm_chain_kernel_name: bad argument");
    GemmPlan plan;
    name[0] = 0;
    *launches = 0;
    if (!chain_pays(n, M, N, K, &plan)) return 0;
    const int len = gemm_chain_kernel_name(plan, name, bytes);
    CACTI_REQUIRE(len >= 0 && (size_t)len < bytes, CACTI_E_INVALID, "gemm_chain_kernel_name: %zu bytes are too few for the name", bytes);
    *launches = plan.cols > 0 ? 2 : 1;
    return 0;
}

CACTI_API int cacti_hip_gemm_f16_chain(int64_t n, int64_t M, int64_t N, int64_t K, const void *const *A, int64_t lda, const void *const *B,
                                       int64_t ldb, float beta, void *C, int64_t ldc, void *stream)
{
    CACTI_REQUIRE(n > 0 && A && B, CACTI_E_INVALID, "gemm_chain: null pointer array or no product");
    for (int64_t z = 0; z < n; z++)
        CACTI_REQUIRE(A[z] && B[z], CACTI_E_INVALID, "gemm_chain: null operand in product %lld", (long long)z);
    bool one = C && beta == 0.f && mult(lda, 8) && mult(ldb, 8) && mult(ldc, 8) && lda >= K && ldb >= N && ldc >= N && lda < kMaxPitch &&
               ldb < kMaxPitch && aligned(C, 16);
    for (int64_t z = 0; z < n && one; z++) one = aligned(A[z], 16) && aligned(B[z], 16);
    GemmPlan plan;
    if (one && chain_pays(n, M, N, K, &plan)) {
        GemmArgs p = {};
        p.M = M; p.N = N; p.K = K; p.alpha = 1.f;
        p.A = (const half_t *)A[0]; p.lda = lda;
        p.B = (const half_t *)B[0]; p.ldb = ldb;
        p.C = (half_t *)C; p.ldc = ldc;
        p.chain = (int)n;
        for (int64_t z = 0; z < n; z++) {
            p.za[z] = (const half_t *)A[z] - p.A;
            p.zb[z] = (const half_t *)B[z] - p.B;
        }
        return gemm_direct_launch(0, 0, p, 1, plan, (hipStream_t)stream);
    }
    for (int64_t z = 0; z < n; z++) {
        const int rc = cacti_hip_gemm_f16(0, 0, M, N, K, 1.f, A[z], lda, B[z], ldb, z ? 1.f : beta, C, ldc, stream);
        if (rc) return rc;
    }
    return 0;
}

static GemmPlan pair_plan(int64_t n, int64_t S, int64_t N, int64_t K, size_t lent = 0)
{
    const bool fits = n >= 1 && n <= kMaxPtrBatch && S > 0 && N > 0 && K > 0 && mult(N, n > 1 ? 64 : 8) && (n == 1 || N >= 4 * 64) &&
                      mult(K, 8) && N < kMaxPitch && K < kMaxPitch;
    return fits ? gemm_plan_pair(S, N, K, (int)n, lent) : GemmPlan{-1, 0, 0, 1, 0};
}

namespace cacti {
bool gemm_pair_pays(int64_t S, int64_t N, int64_t K, int n, size_t lent) { return pair_plan(n, S, N, K, lent).tile >= 0; }
}  // namespace cacti

CACTI_API int cacti_hip_gemm_f16_grads_one_launch(int64_t n, int64_t S, int64_t N, int64_t K) { return pair_plan(n, S, N, K).tile >= 0 ? 1 : 0; }

// whether na f16 values at a and nb at b have one in common
static bool overlap(const void *a, int64_t na, const void *b, int64_t nb)
{
    const uintptr_t p = (uintptr_t)a, q = (uintptr_t)b;
    return na > 0 && nb > 0 && p < q + (uint64_t)nb * sizeof(half_t) && q < p + (uint64_t)na * sizeof(half_t);
}

CACTI_API int cacti_hip_gemm_f16_grads(int64_t n, int64_t S, int64_t N, int64_t K, const void *const *dy, const void *const *W, const void *x,
                                       float beta_x, void *dx, float beta_w, void *const *dW, void *stream)
{
    CACTI_REQUIRE(n > 0 && dy && W && dW && x && dx, CACTI_E_INVALID, "gemm_grads: null pointer or no product");
    for (int64_t z = 0; z < n; z++)
        CACTI_REQUIRE(dy[z] && W[z] && dW[z], CACTI_E_INVALID, "gemm_grads: null operand in product %lld", (long long)z);
    CACTI_REQUIRE((beta_x == 0.f || beta_x == 1.f) && (beta_w == 0.f || beta_w == 1.f), CACTI_E_INVALID, "gemm_grads: beta must be 0 or 1");
    for (int64_t z = 0; z < n; z++) {
        CACTI_REQUIRE(!overlap(dx, S * K, dy[z], S * N) && !overlap(dx, S * K, W[z], N * K), CACTI_E_INVALID,
                      "gemm_grads: dx overlaps an operand of product %lld", (long long)z);
        CACTI_REQUIRE(!overlap(dW[z], N * K, x, S * K) && !overlap(dW[z], N * K, dx, S * K), CACTI_E_INVALID,
                      "gemm_grads: dW of product %lld overlaps x or dx", (long long)z);
        for (int64_t y = 0; y < n; y++)
            CACTI_REQUIRE(!overlap(dW[z], N * K, dy[y], S * N) && !overlap(dW[z], N * K, W[y], N * K) &&
                              (y == z || !overlap(dW[z], N * K, dW[y], N * K)),
                          CACTI_E_INVALID, "gemm_grads: dW of product %lld overlaps a tensor of product %lld", (long long)z, (long long)y);
    }
    const GemmPlan plan = pair_plan(n, S, N, K);
    bool one = plan.tile >= 0 && (n == 1 || beta_x == 0.f) && aligned(x, 16) && aligned(dx, 16);
    if (overlap(dx, S * K, x, S * K)) one = false;         // every weight gradient has read x before dx takes its place
    for (int64_t z = 0; z < n && one; z++) one = aligned(dy[z], 16) && aligned(W[z], 16) && aligned(dW[z], 16);
    if (!one) {
        for (int64_t z = 0; z < n; z += kMaxPtrBatch) {
            const void *xs[kMaxPtrBatch] = {x, x, x, x};
            const int rc = cacti_hip_gemm_f16_batched(1, 0, n - z < kMaxPtrBatch ? n - z : kMaxPtrBatch, N, K, S, 1.f, dy + z, N, xs, K, beta_w,
                                                      dW + z, K, stream);
            if (rc) return rc;
        }
        return cacti_hip_gemm_f16_chain(n, S, K, N, dy, N, W, K, beta_x, dx, K, stream);
    }
    GemmArgs nn = {}, tn = {};
    nn.M = S; nn.N = K; nn.K = N; nn.alpha = 1.f; nn.beta = beta_x;
    nn.A = (const half_t *)dy[0]; nn.lda = N;
    nn.B = (const half_t *)W[0]; nn.ldb = K;
    nn.C = (half_t *)dx; nn.ldc = K;
    nn.chain = (int)n;
    tn.M = N; tn.N = K; tn.K = S; tn.alpha = 1.f; tn.beta = beta_w;
    tn.A = (const half_t *)dy[0]; tn.lda = N;
    tn.B = (const half_t *)x; tn.ldb = K;
    tn.C = (half_t *)dW[0]; tn.ldc = K;
    tn.ztab = n > 1;
    for (int64_t z = 0; z < n; z++) {
        nn.za[z] = tn.za[z] = (const half_t *)dy[z] - nn.A;
        nn.zb[z] = (const half_t *)W[z] - nn.B;
        tn.zc[z] = (half_t *)dW[z] - tn.C;
    }
    return gemm_pair_launch(nn, tn, n, plan, (hipStream_t)stream);
}

CACTI_API int cacti_hip_gemm_f16_strided_batched(int ta, int tb, int64_t nblk, int64_t M, int64_t N,
                                                 int64_t K, float alpha, const void *A, int64_t lda,
                                                 int64_t stride_a, const void *B, int64_t ldb,
                                                 int64_t stride_b, float beta, void *C, int64_t ldc,
                                                 int64_t stride_c, void *stream)
{
    return cacti_hip_gemm_f16_strided_batched_tri(ta, tb, nblk, M, N, K, alpha, A, lda, stride_a, B,
                                                  ldb, stride_b, beta, C, ldc, stride_c, 0, stream);
}

CACTI_API int cacti_hip_gemm_f16(int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha,
                                 const void *A, int64_t lda, const void *B, int64_t ldb, float beta,
                                 void *C, int64_t ldc, void *stream)
{
    return cacti_hip_gemm_f16_strided_batched(ta, tb, 1, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta,
                                              C, ldc, 0, stream);
}

// Column-major C[m x n] = alpha op(a) op(b) + beta C is the row-major product
// C^T[n x m] = op(b)^T op(a)^T, i.e. the row-major kernel with the operands swapped:
// a column-major "N" operand is a row-major transposed one's transpose.
CACTI_API int cacti_hip_gemm_colmajor_f16(int tr_a, int tr_b, int m, int n, int k,
                                          const float *alpha, const void *a, int lda, const void *b,
                                          int ldb, const float *beta, void *c, int ldc, void *stream)
{
    CACTI_REQUIRE(alpha && beta, CACTI_E_INVALID, "gemm_colmajor: null alpha/beta");
    // row-major view: C'[n,m]; first operand op'(b): col-major b (k x n if N) is row-major [n,k]
    // = "transposed" storage of the K x N... expressed through (ta', tb') below.
    // col-major b, tr_b = N: memory holds b[k][n] at n*ldb + k  -> row-major [n][k]: op'(A') = A' (M'=n, K=k): ta' = 0
    // col-major b, tr_b = T: memory holds b[n][k] at k*ldb + n  -> row-major [k][n]: ta' = 1
    // col-major a, tr_a = N: memory a[m][k] at k*lda + m        -> row-major [k][m] = K x N' : tb' = 0
    // col-major a, tr_a = T: memory a[k][m] at m*lda + k        -> row-major [m][k] = N' x K : tb' = 1
    return cacti_hip_gemm_f16(tr_b ? 1 : 0, tr_a ? 1 : 0, n, m, k, *alpha, b, ldb, a, lda, *beta, c,
                              ldc, stream);
}
