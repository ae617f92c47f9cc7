// Shared between the generic GEMM kernel (any alignment) and the 16-byte-aligned fast path.
#pragma once
#include "common.h"

namespace cacti {

// n / d for n < 2^31 by a multiplication: with m = ceil(2^(31 + s) / d) and 2^(s - 1) < d <= 2^s, m d exceeds 2^(31 + s) by
// less than 2^s, so n m exceeds n 2^(31 + s) / d by less than 2^(31 + s) / d.  (A division by a kernel argument is some
// 40 vector instructions, one after another, in front of a workgroup's first load.)
struct FastDiv {
    uint32_t m, shift;
    void set(uint32_t d)
    {
        uint32_t s = 0;
        while ((uint64_t)1 << s < d) s++;
        shift = 31 + s;
        m = (uint32_t)((((uint64_t)1 << shift) + d - 1) / d);
    }
    __host__ __device__ __forceinline__ uint32_t div(uint32_t n) const { return (uint32_t)((uint64_t)n * m >> shift); }
};

// From a workgroup's number to its tile.  Dispatch order i lands on XCD i % 8: each XCD is given a contiguous band of the
// flattened (block of the batch, tile) sequence.  Within a block the tiles are walked in groups of `rows` tile rows x all
// tile columns, row fastest, so that the workgroups resident together on an XCD form a patch of C and share the operand
// panels fetched into its L2.  A pointer-table batch is a handful of whole products that share an operand (the projections
// of one input, the weight gradients against one input): product fastest, so that the workgroups resident together work on
// the same tile of every product and fetch the shared panel once.
struct TileWalk {
    int wgs, nz, ztab, tiles, rows, full, rest, per_group;        // full, rest: tile rows in whole groups, and others
    FastDiv by_tiles, by_nz, by_group, by_rows, by_rest;
    void set(int tiles_m, int tiles_n, int rows_, int64_t nblk, int ztab_)
    {
        tiles = tiles_m * tiles_n;
        nz = (int)nblk;
        wgs = (int)(tiles * nblk);
        ztab = ztab_;
        rows = rows_;
        full = tiles_m / rows * rows;
        by_tiles.set(tiles);
        by_nz.set(nz);
        rest = tiles_m - full;
        per_group = rows * tiles_n;
        by_group.set(per_group);
        by_rows.set(rows);
        by_rest.set(rest ? rest : 1);
    }
    __host__ __device__ __forceinline__ void locate(uint32_t wg, int &tm, int &tn, int &bz) const
    {
        TileWalk w = *this;
#ifdef __HIP_DEVICE_COMPILE__
        // as values, all fetched at once: fields that are read where the control flow first wants them, or by a selected address,
        // cost up to three dependent reads of the argument block, the first of a cache line that nothing has touched yet
        asm volatile("" : "+s"(w.wgs), "+s"(w.nz), "+s"(w.ztab), "+s"(w.tiles), "+s"(w.rows), "+s"(w.full), "+s"(w.rest), "+s"(w.per_group),
                     "+s"(w.by_group.m), "+s"(w.by_group.shift), "+s"(w.by_rows.m), "+s"(w.by_rows.shift), "+s"(w.by_rest.m),
                     "+s"(w.by_rest.shift));
        asm volatile("" : "+s"(w.by_tiles.m), "+s"(w.by_tiles.shift), "+s"(w.by_nz.m), "+s"(w.by_nz.shift));
#endif
        const uint32_t per = (uint32_t)w.wgs >> 3, rem = w.wgs & 7, xcd = wg & 7;
        uint32_t id = xcd * per + (xcd < rem ? xcd : rem) + (wg >> 3);
        bz = 0;
        if (__builtin_expect(w.ztab, 0)) {
            const uint32_t q = w.by_nz.div(id);
            bz = (int)(id - q * w.nz);
            id = q;
        } else if (w.nz > 1) {
            bz = (int)w.by_tiles.div(id);
            id -= (uint32_t)bz * w.tiles;
        }
        const uint32_t group = w.by_group.div(id), in = id - group * w.per_group;
        const int first = (int)group * w.rows;
        const bool whole = first < w.full;
        const FastDiv by = {whole ? w.by_rows.m : w.by_rest.m, whole ? w.by_rows.shift : w.by_rest.shift};
        const uint32_t col = by.div(in);
        tn = (int)col;
        tm = first + (int)(in - col * (whole ? w.rows : w.rest));
    }
};

struct GemmArgs {
    int64_t M, N, K;
    float alpha, beta;
    const half_t *A;
    int64_t lda, sa;
    const half_t *B;
    int64_t ldb, sb;
    half_t *C;
    int64_t ldc, sc;
    int tiles_m, tiles_n;  // (gemm_direct.hip: in `walk` only)
    TileWalk walk;
    // triangular structure of square attention operands (0 = none):
    //  1: only the lower triangle (n <= m) of C is wanted: tiles wholly above it are skipped
    //     and left unwritten;
    //  2: op(A) = A is lower triangular (zero for k > m): the k loop stops at the tile's
    //     last row;
    //  3: op(A) = A^T with A lower triangular (zero for k < m): the k loop starts at the
    //     tile's first row.
    // For 2 and 3 the entries of A above the diagonal must be zero up to the next multiple
    // of 256 columns; beyond that they are never read.
    int tri;
    int pair;             // 1: a workgroup computes tile rows r and tiles_m - 1 - r (tri 2 / 3)
    // 1: B ([K][N] row-major) and C are addressed per block from the 16-byte boundary at or
    // below their first column (column window); set by the entry point when A is 16-byte
    // aligned and B, C are only 8-byte aligned because of their batch stride
    int win;
    // 1: the blocks of the batch are separate arrays: block z starts at A + za[z], B + zb[z],
    // C + zc[z] (element offsets) instead of z times the batch strides; at most kMaxPtrBatch blocks
    int ztab;
    int64_t za[4], zb[4], zc[4];
    // part: the product in parts of K of split_tiles k tiles each, whose fp32 sums go to part[part][M][ldp]
    int split_tiles;
    float *part;
    int64_t ldp;
    // chain > 1: the sum of that many products A + za[z], B + zb[z], rounded to f16 with what the ones before came to (beta 0)
    int chain;
    int odd;              // C of any alignment and N
    int any;              // A and B of any alignment (strided operands with rows of 8 elements and more)
};
constexpr int kMaxPtrBatch = 4;
constexpr int kTriPad = 256;

// how gemm_direct_launch cuts a product whose operands are 16-byte aligned: tile shapes as in gemm_direct.hip
struct GemmPlan {
    int tile, rest;      // shape of the (first) launch; of the second
    int64_t cols;        // > 0: columns of the first launch, the rest go to a second
    int split;           // parts of K
    double us;           // what it is expected to take
};
// nz: products of this shape in the launch; lent: the largest workspace that the parts of one may take (0: it stays whole)
GemmPlan gemm_plan(int64_t M, int64_t N, int64_t K, int64_t nz, size_t lent);
inline int64_t gemm_part_pitch(int64_t N) { return (N + 3) / 4 * 4; }            // GemmArgs::ldp
inline size_t gemm_parts_bytes(int64_t M, int64_t N, int split) { return (size_t)split * (size_t)M * (size_t)gemm_part_pitch(N) * sizeof(float); }
GemmPlan gemm_plan_parts(int64_t M, int64_t N, int64_t K, int parts);       // in exactly that many parts, 2 .. 8 (tile < 0: K has none)
GemmPlan gemm_plan_chain(int64_t M, int64_t N, int64_t K, int chain);       // chain <= kMaxPtrBatch products that add up
// the gradients of n products x W_i^T, x [S,K], W_i [N,K], all in one launch (tile < 0: no better than two, the input gradient of a
// single product among them with `lent` bytes for parts of K)
GemmPlan gemm_plan_pair(int64_t S, int64_t N, int64_t K, int n, size_t lent);
bool gemm_pair_pays(int64_t S, int64_t N, int64_t K, int n, size_t lent);
// cacti_hip_gemm_f16_ws that asks for no more than `most` bytes, in fewer parts or without a copy if need be
int gemm_f16_within(size_t most, int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha, const void *A, int64_t lda, const void *B, int64_t ldb,
                    float beta, void *C, int64_t ldc, void *ws, size_t ws_bytes, size_t *ws_need, hipStream_t st);
// the parts of K that it takes of whole matrices that begin on 16 bytes (1: whole, or rows between 16-byte boundaries)
int gemm_parts_within(size_t most, int ta, int tb, int64_t M, int64_t N, int64_t K, bool acc);
GemmPlan gemm_plan_any(int64_t M, int64_t N, int64_t K, size_t lent);        // for GemmArgs::any (with parts of K)
void gemm_tile_dims(int tile, int64_t *bm, int64_t *bn);
// the kernel of the plan's (first) launch as a profiler prints it; returns what snprintf does
int gemm_kernel_name(int ta, int tb, const GemmPlan &plan, char *name, size_t bytes);
int gemm_chain_kernel_name(const GemmPlan &plan, char *name, size_t bytes);

// Products of operands whose rows are at least 8-byte aligned (align = 4; 8: 16-byte aligned), with a triangular operand or
// a column window among them.
int gemm_mfma_launch(int ta, int tb, const GemmArgs &p, int64_t nblk, int align, hipStream_t st);

// Products of 16-byte aligned operands, cut by `plan` (p.part lent for its parts; p.odd: C of any alignment and N; tri and win
// are not for these).
int gemm_direct_launch(int ta, int tb, const GemmArgs &p, int64_t nblk, const GemmPlan &plan, hipStream_t st);

int gemm_pair_launch(const GemmArgs &nn, const GemmArgs &tn, int64_t nblk, const GemmPlan &plan, hipStream_t st);

// tile rows per group of the walk of a launch of tiles_m x tiles_n tiles of bm x bn
int gemm_walk_rows(int tiles_m, int tiles_n, int bm, int bn, int64_t nblk);

int gemm_repack(const half_t *const src[2], half_t *const dst[2], const int64_t rows[2], const int64_t cols[2],
                const int64_t ld[2], hipStream_t st);

// C = f16(alpha A B^T) with K <= 128 (attention scores): A [M,K], B [N,K] row-major, rows
// 8-byte aligned, K % 4 == 0, beta = 0, tri 0 or 1
int gemm_nt_smallk_launch(const GemmArgs &p, int64_t nblk, hipStream_t st);

// C[M,N] = f16(alpha A B^T) for 1 <= M <= 4: a stream over B ([N,K] row-major, rows 16-byte
// aligned, K % 8 == 0), beta = 0; A rows 16-byte aligned
int gemm_skinny_nt_launch(int64_t M, int64_t N, int64_t K, float alpha, const half_t *A, int64_t lda,
                          const half_t *B, int64_t ldb, half_t *C, int64_t ldc, hipStream_t st);

// The decoding kernels of gemm_skinny.hip as the cached forward pass uses them (1 to 4 rows of K <= 8192 elements,
// K % 8 == 0, everything 16-byte aligned).  The rows are rms_norm(x or f16(x + x2), w_norm); with tok, row m of x is row
// tok[m] of a table of `vocab` rows (an id out of range raises *status to m + 1).
struct RowSource {
    const void *x, *x2, *w_norm;
    float eps;
    const uint16_t *tok;
    int64_t vocab;
    int *status;
};
int rows_qkv_launch(int64_t M, int64_t H, int64_t Dh, const RowSource &x, void *sum_out, const void *Wq, const void *Wk, const void *Wv,
                    const void *cos16, const void *sin16, void *q_rot, void *k_cache_rows, void *v_cache_rows, hipStream_t st);
int rows_gate_launch(int64_t M, int64_t N, int64_t K, const RowSource &x, void *sum_out, const void *B, const void *B_mul, void *C,
                     hipStream_t st);
int rows_norm_launch(int64_t M, int64_t N, int64_t K, const RowSource &x, const void *B, void *C, hipStream_t st);
// logit = rows B^T and the arg max of each row in out_tok; the last row's token is added to in_tok[pos] where pos >= 0
size_t rows_head_scratch_bytes(int64_t M, int64_t N);
int rows_head_launch(int64_t M, int64_t N, int64_t K, const RowSource &x, const void *B, void *logit, void *scratch, void *out_tok,
                     void *in_tok, int64_t pos, hipStream_t st);

}  // namespace cacti
