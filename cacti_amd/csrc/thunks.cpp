#include "thunks.h"

#include "common.h"
#include "gemm_internal.h"
#include "rmsnorm.h"

namespace cacti {
namespace {

inline void *S(Ctx &c) { return (void *)c.stream(); }

#define TY_REQUIRE(cond, ...) CACTI_REQUIRE(cond, CACTI_E_INVALID, __VA_ARGS__)

// ---------------------------------------------------------------------------
// copy (the memcpy adjoint of Add / Identity, src/thunk/op.rs:1529-1534, 5474-5729)
struct CopySpec : ThunkSpec {
    const char *name() const override { return "copy"; }
    int arity() const override { return 1; }
    bool is_copy() const override { return true; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        o = {a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        if (acc & 1) {
            TY_REQUIRE(aty[0].dtype == F16, "copy: accumulate is f16 only");
            return cacti_hip_add_f16(aty[0].numel(), o[0], a[0], o[0], S(c));
        }
        return cacti_hip_memcpy_async(o[0], a[0], aty[0].bytes(), S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        return c.adj_add({e.args[0]}, make_copy(), {dy[0]});
    }
};

// ---------------------------------------------------------------------------
// y = a + b (AddFutThunkSpec src/thunk/op.rs:1480-1535); both adjoints are copies of dy
struct AddSpec : ThunkSpec {
    const char *name() const override { return "add"; }
    int arity() const override { return 2; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0] == a[1] && a[0].dtype == F16, "add: operands must be equal f16 shapes");
        o = {a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        TY_REQUIRE(!(acc & 1), "add: accumulate mode not staged on this path");
        return cacti_hip_add_f16(aty[0].numel(), a[0], a[1], o[0], S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        int rc = c.adj_add({e.args[0]}, make_copy(), {dy[0]});
        if (rc) return rc;
        return c.adj_add({e.args[1]}, make_copy(), {dy[0]});
    }
};

// ---------------------------------------------------------------------------
// Embedding (OuterSelectFutThunkSpec src/thunk/op.rs:1229-1314) and its scatter-add adjoint
struct EmbedBwdSpec : ThunkSpec {
    int64_t V;
    explicit EmbedBwdSpec(int64_t v) : V(v) {}
    const char *name() const override { return "embed_bwd"; }
    int arity() const override { return 2; }                       // (tok, dy) -> dW
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == U16 && a[1].dtype == F16 && a[1].shape.size() == 2,
                   "embed_bwd: (tok u16, dy f16 [S,D]) expected");
        o = {CellType({V, a[1].shape[1]}, F16)};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        return cacti_hip_embed_bwd(V, aty[1].shape[1], aty[1].shape[0], a[0], a[1], o[0], acc & 1,
                                   S(c));
    }
};

struct EmbedSpec : ThunkSpec {
    const char *name() const override { return "embed"; }
    int arity() const override { return 2; }                       // (W, tok) -> y
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == F16 && a[0].shape.size() == 2 && a[1].dtype == U16,
                   "embed: (W f16 [V,D], tok u16) expected");
        o = {CellType({a[1].numel(), a[0].shape[1]}, F16)};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t, void *, size_t) const override
    {
        return cacti_hip_embed_fwd(aty[0].shape[0], aty[0].shape[1], a[0], aty[1].numel(), a[1],
                                   o[0], c.status_ptr(), S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        const int64_t V = c.cell(e.args[0]).ty.shape[0];
        return c.adj_add({e.args[0]}, std::unique_ptr<ThunkSpec>(new EmbedBwdSpec(V)),
                         {e.args[1], dy[0]});
    }
};

// ---------------------------------------------------------------------------
// RMSNorm (rms_norm closure src/librarium/llama.rs:442-451) and its fused adjoint
struct RmsNormBwdSpec : ThunkSpec {
    float eps;
    explicit RmsNormBwdSpec(float e) : eps(e) {}
    const char *name() const override { return "rms_norm_bwd"; }
    int arity() const override { return 3; }                       // (x, w, dy) -> dx, partial rows of dw
    int nout() const override { return 2; }
    static CellType parts(const CellType &x)
    {
        const size_t bytes = cacti_hip_rms_norm_bwd_workspace(x.shape[0], x.shape[1]);
        return CellType({(int64_t)(bytes / sizeof(float)) / x.shape[1], x.shape[1]}, F32);
    }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0] == a[2] && a[0].shape.size() == 2 && a[1].numel() == a[0].shape[1],
                   "rms_norm_bwd: shape mismatch");
        o = {a[0], parts(a[0])};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &oty,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        return rms_norm_bwd_parts(aty[0].shape[0], aty[0].shape[1], a[0], a[1], eps, a[2], o[0], acc & 1, o[1], oty[1].bytes(), c.stream());
    }
};

// The sums of the partial rows of several norms, each an output like `ty[i]`
struct RmsNormDwSpec : ThunkSpec {
    std::vector<CellType> ty;
    explicit RmsNormDwSpec(std::vector<CellType> t) : ty(std::move(t)) {}
    const char *name() const override { return "rms_norm_dw"; }
    int arity() const override { return (int)ty.size(); }
    int nout() const override { return (int)ty.size(); }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        for (size_t i = 0; i < a.size(); i++)
            TY_REQUIRE(a[i] == a[0] && a[i].dtype == F32 && a[i].shape.size() == 2 && ty[i].dtype == F16 && ty[i].numel() == a[i].shape[1],
                       "rms_norm_dw: shape mismatch");
        o = ty;
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        return rms_norm_dw_sums((int)ty.size(), aty[0].shape[0], aty[0].shape[1], a, o, acc, c.stream());
    }
    int pieces() const override { return (int)ty.size(); }
    std::unique_ptr<ThunkSpec> piece(int i, const std::vector<CellPtr> &args, std::vector<CellPtr> *of) const override
    {
        *of = {args[(size_t)i]};
        return std::unique_ptr<ThunkSpec>(new RmsNormDwSpec({ty[(size_t)i]}));
    }
    // launches of another number of sums are others; ",acc" and the outputs that are added to, in hexadecimal
    std::string key(const std::vector<CellType> &aty, uint32_t acc) const override
    {
        char buf[96], mode[16] = "";
        if (acc) snprintf(mode, sizeof(mode), ",acc%x", acc);
        snprintf(buf, sizeof(buf), "rms_norm_dw[%lldx%lld%s]x%zu", (long long)aty[0].shape[0], (long long)aty[0].shape[1], mode, ty.size());
        return buf;
    }
};

// dx (+)= and the partial rows of dw now, their sum with those of the norms to come
int norm_adjoint(Ctx &c, float eps, CellPtr x, CellPtr w, CellPtr dy)
{
    const bool sum = c.adj_of(w) != 0;
    const CellPtr rows = c.cell_new(RmsNormBwdSpec::parts(c.cell(x).ty), false, "dw rows");
    const int rc = c.adj_add({x}, std::unique_ptr<ThunkSpec>(new RmsNormBwdSpec(eps)), {x, w, dy}, {rows}, sum);
    return rc || !sum ? rc : c.adj_sum_later(w, rows);
}

struct RmsNormSpec : ThunkSpec {
    float eps;
    explicit RmsNormSpec(float e) : eps(e) {}
    const char *name() const override { return "rms_norm"; }
    int arity() const override { return 2; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == F16 && a[1].dtype == F16 && a[0].shape.size() == 2 &&
                       a[1].numel() == a[0].shape[1],
                   "rms_norm: (x f16 [N,D], w f16 [D]) expected");
        o = {a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t, void *, size_t) const override
    {
        return cacti_hip_rms_norm_fwd(aty[0].shape[0], aty[0].shape[1], a[0], a[1], eps, o[0], S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        return norm_adjoint(c, eps, e.args[0], e.args[1], dy[0]);
    }
};

// x = a + b followed by y = rms_norm(x, w) as one launch with both outputs (the residual add
// always feeds a norm: llama.rs:512-516 and :532 -> the next layer's :474 / the head's :536).
// The adjoint is the two thunks' rules in their reverse order: the norm's adjoint accumulates
// into the adjoint of x, which the add's two memcpy adjoints then hand on.
struct AddRmsNormSpec : ThunkSpec {
    float eps;
    explicit AddRmsNormSpec(float e) : eps(e) {}
    const char *name() const override { return "add_rms_norm"; }
    int arity() const override { return 3; }                       // (a, b, w) -> x, y
    int nout() const override { return 2; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0] == a[1] && a[0].dtype == F16 && a[2].dtype == F16 && a[0].shape.size() == 2 &&
                       a[2].numel() == a[0].shape[1],
                   "add_rms_norm: (a, b f16 [N,D], w f16 [D]) expected");
        o = {a[0], a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        TY_REQUIRE(acc == 0, "add_rms_norm: accumulate mode not staged on this path");
        return cacti_hip_add_rms_norm_fwd(aty[0].shape[0], aty[0].shape[1], a[0], a[1], a[2], eps, o[0],
                                          o[1], S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        if (dy[1]) {
            const int rc = norm_adjoint(c, eps, e.outs[0], e.args[2], dy[1]);
            if (rc) return rc;
        }
        if (!c.adj_written(e.outs[0])) return 0;
        const CellPtr dx = c.adj_of(e.outs[0]);
        int rc = c.adj_add({e.args[0]}, make_copy(), {dx});
        if (rc) return rc;
        return c.adj_add({e.args[1]}, make_copy(), {dx});
    }
};

// ---------------------------------------------------------------------------
// MatrixMulThunkSpec src/thunk/op.rs:4284-4368 (2-d) and BlockMatrixMulThunkSpec :4719-4918
// on [R, H*C] tensors (the reference's [B,S,H,C] with B = 1, flattened) whose H per-head
// blocks are addressed by stride; H = 0 means one plain matrix.
//
// `causal` marks the two products of causal attention (scores = a Q K^T whose upper
// triangle the mask discards: CAUSAL_OUT; P V with P lower triangular: CAUSAL_A) so that
// the discarded half is not computed; the adjoint rules carry the structure along
// (dP = dO V^T is only needed below the diagonal; dV = P^T dO, dQ = a dS K, dK = a dS^T Q
// have a triangular first operand).
enum { CAUSAL_NONE = 0, CAUSAL_OUT = 1, CAUSAL_A = 2 };
struct MatMulSpec : ThunkSpec {
    bool ta, tb;
    int64_t nblk;
    bool blocked;
    float alpha;
    int causal;
    bool lend = false;               // a workspace (Ctx::product_scratch) for parts of K and operands of any alignment, where it asks for one
    MatMulSpec(bool a, bool b, float al, int64_t h, int cz = CAUSAL_NONE)
        : ta(a), tb(b), nblk(h), blocked(h > 0), alpha(al), causal(cz) {}
    const char *name() const override { return blocked ? "block_matmul" : "matmul"; }
    int arity() const override { return 2; }
    struct Dims { int64_t H, M, N, K, lda, sa, ldb, sb, ldc, sc; };
    int dims(const std::vector<CellType> &a, Dims &d) const
    {
        TY_REQUIRE(a[0].dtype == F16 && a[1].dtype == F16 && a[0].shape.size() == 2 &&
                       a[1].shape.size() == 2,
                   "%s: f16 operands of rank 2 expected", name());
        d.H = blocked ? nblk : 1;
        TY_REQUIRE(a[0].shape[1] % d.H == 0 && a[1].shape[1] % d.H == 0,
                   "block_matmul: row length not divisible by the block count");
        const int64_t ra = a[0].shape[0], ca = a[0].shape[1] / d.H;
        const int64_t rb = a[1].shape[0], cb = a[1].shape[1] / d.H;
        d.M = ta ? ca : ra;
        d.K = ta ? ra : ca;
        const int64_t kb = tb ? cb : rb;
        d.N = tb ? rb : cb;
        TY_REQUIRE(kb == d.K, "%s: inner dimensions %lld and %lld differ", name(), (long long)d.K,
                   (long long)kb);
        d.lda = d.H * ca; d.sa = ca;
        d.ldb = d.H * cb; d.sb = cb;
        d.ldc = d.H * d.N; d.sc = d.N;
        return 0;
    }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        Dims d;
        int rc = dims(a, d);
        if (rc) return rc;
        o = {CellType({d.M, d.H * d.N}, F16)};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        Dims d;
        int rc = dims(aty, d);
        if (rc) return rc;
        if (lend && !blocked) {
            size_t need = 0;
            void *ws = nullptr;
            auto product = [&]() {
                return gemm_f16_within(Ctx::kProductScratch, ta, tb, d.M, d.N, d.K, alpha, a[0], d.lda, a[1], d.ldb, (acc & 1) ? 1.f : 0.f,
                                       o[0], d.ldc, ws, need, &need, c.stream());
            };
            if ((rc = product()) || need == 0) return rc;
            if ((ws = c.product_scratch(need))) return product();
        }
        const int tri = causal == CAUSAL_OUT ? 1 : causal == CAUSAL_A ? (ta ? 3 : 2) : 0;
        return cacti_hip_gemm_f16_strided_batched_tri(ta, tb, d.H, d.M, d.N, d.K, alpha, a[0],
                                                      d.lda, d.sa, a[1], d.ldb, d.sb,
                                                      (acc & 1) ? 1.f : 0.f, o[0], d.ldc, d.sc, tri,
                                                      S(c));
    }
    std::string key(const std::vector<CellType> &aty, uint32_t acc) const override
    {
        Dims d;
        if (dims(aty, d)) return name();
        // ",parts2": in two parts of K, a launch of the parts and one of their sum
        char buf[128], parts[16] = "";
        const int split = lend && !blocked ? gemm_parts_within(Ctx::kProductScratch, ta, tb, d.M, d.N, d.K, acc & 1) : 1;
        if (split > 1) snprintf(parts, sizeof(parts), ",parts%d", split);
        snprintf(buf, sizeof(buf), "%s[%c%c,%lldx%lldx%lldx%lld%s%s]", name(), ta ? 'T' : 'N',
                 tb ? 'T' : 'N', (long long)d.H, (long long)d.M, (long long)d.N, (long long)d.K,
                 (acc & 1) ? ",acc" : "", parts);
        return buf;
    }
    std::unique_ptr<ThunkSpec> mm(bool x, bool y, int cz = CAUSAL_NONE) const
    {
        return std::unique_ptr<ThunkSpec>(new MatMulSpec(x, y, alpha, nblk, cz));
    }
    // the four transposition cases of pop_adj, src/thunk/op.rs:4335-4367 / :4882-4912:
    // arg_adj[1] first, then arg_adj[0], both carrying o_scale
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        const CellPtr A = e.args[0], B = e.args[1], G = dy[0];
        int rc;
        if (causal == CAUSAL_OUT) {              // C = a A B^T, only tril(C) is used: G = tril
            TY_REQUIRE(!ta && tb, "causal scores product must be A B^T");
            if ((rc = c.adj_add({B}, mm(true, false, CAUSAL_A), {G, A}))) return rc;   // G^T A
            return c.adj_add({A}, mm(false, false, CAUSAL_A), {G, B});                  // G B
        }
        if (causal == CAUSAL_A) {                // C = A B with A = tril
            TY_REQUIRE(!ta && !tb, "causal probability product must be A B");
            if ((rc = c.adj_add({B}, mm(true, false, CAUSAL_A), {A, G}))) return rc;   // A^T G
            return c.adj_add({A}, mm(false, true, CAUSAL_OUT), {G, B});                 // tril(G B^T)
        }
        if (!ta && !tb) {
            if ((rc = c.adj_add({B}, mm(true, false), {A, G}))) return rc;      // A^T G
            return c.adj_add({A}, mm(false, true), {G, B});                      // G B^T
        }
        if (!ta && tb) {
            if ((rc = c.adj_add({B}, mm(true, false), {G, A}))) return rc;      // G^T A
            return c.adj_add({A}, mm(false, false), {G, B});                     // G B
        }
        if (ta && !tb) {
            if ((rc = c.adj_add({B}, mm(false, false), {A, G}))) return rc;     // A G
            return c.adj_add({A}, mm(false, true), {B, G});                      // B G^T
        }
        if ((rc = c.adj_add({B}, mm(true, true), {G, A}))) return rc;           // G^T A^T
        return c.adj_add({A}, mm(true, true), {B, G});                           // B^T G^T
    }
};

// ---------------------------------------------------------------------------
// Several products of one shape that share an operand, as one thunk and one launch (a pointer-array batch,
// cacti_hip_gemm_f16_batched: the shape of the reference's cublasGemmBatchedEx call,
// cacti_gpu_cu_ffi/src/lib.rs:793-885).  The reference stages the query, key and value projections of a layer
// (and the gate and up projections) as separate matmul thunks on the same input (src/librarium/llama.rs:
// 478-497); each output here is summed over the same values in the same order as in a launch of its own (the tiles
// may be others), so the results are those of the separate thunks bit for bit, and the adjoint stages what their
// adjoints would have staged, in their order: the weight gradients (one grouped thunk), then the input gradients (one thunk and
// launch as well, cacti_hip_gemm_f16_chain: they accumulate into one cell, last product first, as the reverse sweep over
// separate thunks meets them, with a rounding behind each).
constexpr int kMaxGroup = 4;

// dW_i = dy_i^T x: (dy_1 .. dy_n, x) -> (dW_1 .. dW_n)
struct WgradNSpec : ThunkSpec {
    int n;
    explicit WgradNSpec(int n_) : n(n_) {}
    const char *name() const override { return "matmul"; }
    int arity() const override { return n + 1; }
    int nout() const override { return n; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(n >= 2 && n <= kMaxGroup, "grouped weight gradients: 2 .. %d products", kMaxGroup);
        for (int i = 0; i <= n; i++)
            TY_REQUIRE(a[i].dtype == F16 && a[i].shape.size() == 2 && a[i].shape[0] == a[n].shape[0] &&
                           (i == n || a[i] == a[0]),
                       "grouped weight gradients: (dy f16 [S,N] x n, x f16 [S,K]) expected");
        o.assign(n, CellType({a[0].shape[1], a[n].shape[1]}, F16));
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        const int64_t Sq = aty[0].shape[0], N = aty[0].shape[1], K = aty[n].shape[1];
        const uint32_t all = (1u << n) - 1;
        if ((acc & all) != 0 && (acc & all) != all) {          // mixed modes: one after the other
            for (int i = 0; i < n; i++) {
                const int rc = cacti_hip_gemm_f16(1, 0, N, K, Sq, 1.f, a[i], N, a[n], K, ((acc >> i) & 1) ? 1.f : 0.f,
                                                  o[i], K, S(c));
                if (rc) return rc;
            }
            return 0;
        }
        const void *A[kMaxGroup], *B[kMaxGroup];
        void *C[kMaxGroup];
        for (int i = 0; i < n; i++) {
            A[i] = a[i];
            B[i] = a[n];
            C[i] = o[i];
        }
        return cacti_hip_gemm_f16_batched(1, 0, n, N, K, Sq, 1.f, A, N, B, K, (acc & 1) ? 1.f : 0.f, C, K, S(c));
    }
    int pieces() const override { return n; }
    std::unique_ptr<ThunkSpec> piece(int i, const std::vector<CellPtr> &a, std::vector<CellPtr> *in) const override
    {
        *in = {a[(size_t)i], a[(size_t)n]};
        return make_matmul(true, false, 1.f);
    }
    std::string key(const std::vector<CellType> &aty, uint32_t acc) const override
    {
        char buf[128];
        snprintf(buf, sizeof(buf), "matmul[TN,1x%lldx%lldx%lld%s]x%d", (long long)aty[0].shape[1],
                 (long long)aty[n].shape[1], (long long)aty[0].shape[0], (acc & 1) ? ",acc" : "", n);
        return buf;
    }
};

// dx = dy_1 W_1 + .. + dy_n W_n, each product rounded to f16 with the sum of the ones before it:
// (dy_1 .. dy_n, W_1 .. W_n) -> dx
struct DgradNSpec : ThunkSpec {
    int n;
    explicit DgradNSpec(int n_) : n(n_) {}
    const char *name() const override { return "matmul"; }
    int arity() const override { return 2 * n; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(n >= 2 && n <= kMaxGroup, "chained input gradients: 2 .. %d products", kMaxGroup);
        for (int i = 0; i < n; i++)
            TY_REQUIRE(a[i].dtype == F16 && a[i].shape.size() == 2 && a[i] == a[0] && a[n + i] == a[n] && a[n].dtype == F16 &&
                           a[n].shape.size() == 2 && a[n].shape[0] == a[0].shape[1],
                       "chained input gradients: (dy f16 [S,N] x n, W f16 [N,K] x n) expected");
        o.assign(1, CellType({a[0].shape[0], a[n].shape[1]}, F16));
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        const int64_t Sq = aty[0].shape[0], N = aty[0].shape[1], K = aty[n].shape[1];
        return cacti_hip_gemm_f16_chain(n, Sq, K, N, a, N, a + n, K, (acc & 1) ? 1.f : 0.f, o[0], K, S(c));
    }
    int pieces() const override { return n; }
    int piece_out(int) const override { return 0; }
    std::unique_ptr<ThunkSpec> piece(int i, const std::vector<CellPtr> &a, std::vector<CellPtr> *in) const override
    {
        *in = {a[(size_t)i], a[(size_t)(n + i)]};
        return make_matmul(false, false, 1.f);
    }
    std::string key(const std::vector<CellType> &aty, uint32_t acc) const override
    {
        char buf[128];
        snprintf(buf, sizeof(buf), "matmul[NN,1x%lldx%lldx%lld%s]x%d", (long long)aty[0].shape[0], (long long)aty[n].shape[1],
                 (long long)aty[0].shape[1], (acc & 1) ? ",acc" : "", n);
        return buf;
    }
};

// All gradients of n products x W_i^T in one launch: (dy_1 .. dy_n, W_1 .. W_n, x) -> (dx, dW_1 .. dW_n), dx as above
struct GradsNSpec : ThunkSpec {
    int n;
    explicit GradsNSpec(int n_) : n(n_) {}
    const char *name() const override { return "matmul"; }
    int arity() const override { return 2 * n + 1; }
    int nout() const override { return n + 1; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(n >= 1 && n <= kMaxGroup, "gradients of products: 1 .. %d of them", kMaxGroup);
        const CellType &x = a[(size_t)(2 * n)];
        for (int i = 0; i < n; i++)
            TY_REQUIRE(a[i].dtype == F16 && a[i].shape.size() == 2 && a[i] == a[0] && a[n + i] == a[n] && a[n].dtype == F16 &&
                           a[n].shape.size() == 2 && a[n].shape[0] == a[0].shape[1] && x.dtype == F16 && x.shape.size() == 2 &&
                           x.shape[0] == a[0].shape[0] && x.shape[1] == a[n].shape[1],
                       "gradients of products: (dy f16 [S,N] x n, W f16 [N,K] x n, x f16 [S,K]) expected");
        o.assign((size_t)(n + 1), a[n]);
        o[0] = x;
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        const int64_t Sq = aty[0].shape[0], N = aty[0].shape[1], K = aty[n].shape[1];
        const uint32_t all = (1u << n) - 1, dw = acc >> 1 & all;
        if (dw != 0 && dw != all) {                            // mixed modes: one after the other
            for (int i = 0; i < n; i++) {
                const int rc = cacti_hip_gemm_f16(1, 0, N, K, Sq, 1.f, a[i], N, a[2 * n], K, ((dw >> i) & 1) ? 1.f : 0.f, o[1 + i], K, S(c));
                if (rc) return rc;
            }
            return cacti_hip_gemm_f16_chain(n, Sq, K, N, a, N, a + n, K, (acc & 1) ? 1.f : 0.f, o[0], K, S(c));
        }
        return cacti_hip_gemm_f16_grads(n, Sq, N, K, a, a + n, a[2 * n], (acc & 1) ? 1.f : 0.f, o[0], dw ? 1.f : 0.f, o + 1, S(c));
    }
    int pieces() const override { return 2 * n; }
    int piece_out(int i) const override { return i < n ? 1 + i : 0; }
    std::unique_ptr<ThunkSpec> piece(int i, const std::vector<CellPtr> &a, std::vector<CellPtr> *in) const override
    {
        *in = {a[(size_t)(i % n)], a[(size_t)(i < n ? 2 * n : i)]};
        return make_matmul(i < n, false, 1.f);
    }
    // ",acc" and the bits of the outputs (dx, dW_1 ..) that are added to, in hexadecimal
    std::string key(const std::vector<CellType> &aty, uint32_t acc) const override
    {
        char buf[128], mode[16] = "";
        if (acc) snprintf(mode, sizeof(mode), ",acc%x", acc);
        snprintf(buf, sizeof(buf), "matmul_grads[%lldx%lldx%lld%s]x%d", (long long)aty[0].shape[0], (long long)aty[0].shape[1],
                 (long long)aty[n].shape[1], mode, n);
        return buf;
    }
};
// whether the gradients of n products x W_i^T are one launch (apart, a single one's input gradient is lent a workspace)
static bool one_launch(const CellType &dy, const CellType &w, int n)
{
    return gemm_pair_pays(dy.shape[0], dy.shape[1], w.shape[1], n, n > 1 ? 0 : Ctx::kProductScratch);
}
// the gradients of y_i = x W_i^T for the dy in `dy`, last product first, as one thunk if one launch of them pays; *staged: it did
static int stage_grads(Ctx &c, CellPtr x, const std::vector<CellPtr> &ws, const std::vector<CellPtr> &dy, bool *staged)
{
    const int n = (int)ws.size();
    *staged = one_launch(c.cell(dy[0]).ty, c.cell(ws[0]).ty, n);
    if (!*staged) return 0;
    std::vector<CellPtr> primals = {x}, in(dy.rbegin(), dy.rend());
    primals.insert(primals.end(), ws.rbegin(), ws.rend());
    in.insert(in.end(), ws.rbegin(), ws.rend());
    in.push_back(x);
    return c.adj_add(primals, std::unique_ptr<ThunkSpec>(new GradsNSpec(n)), in);
}

// y_i = x W_i^T: (x, W_1 .. W_n) -> (y_1 .. y_n)
struct ProjNSpec : ThunkSpec {
    int n;
    bool group_adj;                  // the gradients grouped as well
    explicit ProjNSpec(int n_, bool ga = true) : n(n_), group_adj(ga) {}
    const char *name() const override { return "matmul"; }
    int arity() const override { return n + 1; }
    int nout() const override { return n; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(n >= 2 && n <= kMaxGroup, "grouped projections: 2 .. %d products", kMaxGroup);
        for (int i = 0; i <= n; i++)
            TY_REQUIRE(a[i].dtype == F16 && a[i].shape.size() == 2 && a[i].shape[1] == a[0].shape[1] &&
                           (i == 0 || a[i] == a[1]),
                       "grouped projections: (x f16 [S,K], W f16 [N,K] x n) expected");
        o.assign(n, CellType({a[0].shape[0], a[1].shape[0]}, F16));
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        TY_REQUIRE(acc == 0, "grouped projections: accumulate mode not staged on this path");
        const int64_t Sq = aty[0].shape[0], K = aty[0].shape[1], N = aty[1].shape[0];
        const void *A[kMaxGroup], *B[kMaxGroup];
        void *C[kMaxGroup];
        for (int i = 0; i < n; i++) {
            A[i] = a[0];
            B[i] = a[1 + i];
            C[i] = o[i];
        }
        return cacti_hip_gemm_f16_batched(0, 1, n, Sq, N, K, 1.f, A, K, B, K, 0.f, C, N, S(c));
    }
    int pieces() const override { return n; }
    std::unique_ptr<ThunkSpec> piece(int i, const std::vector<CellPtr> &a, std::vector<CellPtr> *in) const override
    {
        *in = {a[0], a[(size_t)(1 + i)]};
        return make_matmul(false, true, 1.f);
    }
    std::string key(const std::vector<CellType> &aty, uint32_t) const override
    {
        char buf[128];
        snprintf(buf, sizeof(buf), "matmul[NT,1x%lldx%lldx%lld]x%d", (long long)aty[0].shape[0],
                 (long long)aty[1].shape[0], (long long)aty[0].shape[1], n);
        return buf;
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        const CellPtr x = e.args[0];
        bool all = group_adj;
        for (int i = 0; i < n; i++) all = all && dy[i];
        int rc;
        if (all) {
            std::vector<CellPtr> ws(e.args.begin() + 1, e.args.end()), in(dy.begin(), dy.begin() + n);
            bool staged = false;
            if ((rc = stage_grads(c, x, ws, in, &staged)) || staged) return rc;
            in.push_back(x);
            if ((rc = c.adj_add(ws, std::unique_ptr<ThunkSpec>(new WgradNSpec(n)), in))) return rc;
            std::vector<CellPtr> chain(dy.rend() - n, dy.rend());
            chain.insert(chain.end(), ws.rbegin(), ws.rend());
            return c.adj_add({x}, std::unique_ptr<ThunkSpec>(new DgradNSpec(n)), chain);
        }
        for (int i = n - 1; i >= 0; i--) {
            if (!dy[i]) continue;
            const CellPtr W = e.args[1 + i];
            if ((rc = c.adj_add({W}, std::unique_ptr<ThunkSpec>(new MatMulSpec(true, false, 1.f, 0)), {dy[i], x})))
                return rc;                                                     // G^T A
            if ((rc = c.adj_add({x}, std::unique_ptr<ThunkSpec>(new MatMulSpec(false, false, 1.f, 0)), {dy[i], W})))
                return rc;                                                     // G B
        }
        return 0;
    }
};

// ---------------------------------------------------------------------------
// y = x W^T of a layer: its gradients are one thunk where one launch of both pays (`one`), and it and its input gradient are lent a
// workspace, the sums of few rows over a long K being the work of a few CUs otherwise, and rows between 16-byte boundaries (an FFN
// width that is no multiple of 8: 512 x 1024 x 2815 129 -> 21 us) loaded an element at a time: the head's
// input gradient of 48 x 256 (vocabulary 21480) 66 -> 16 us, 80 x 1024 (29848) 93 -> 21, 112 x 768 (31600) 114 -> 22, 160 x 2048 (31432)
// 156 -> 51, 611 x 1024 (8192) 32 -> 23, 2048 x 3200 (32000) 352 -> 316, and cycles of one layer around them 240 -> 200, 360 -> 283,
// 356 -> 266, 659 -> 527, 311 -> 299, 2906 -> 2849.  (Products that have a grouped form are lent
// none: alone, they have the group's bits.  So has the input gradient where the launch of both would pay.)
struct LinearSpec : MatMulSpec {
    bool one;
    explicit LinearSpec(bool o) : MatMulSpec(false, true, 1.f, 0), one(o) { lend = true; }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        bool staged = false;
        int rc = one ? stage_grads(c, e.args[0], {e.args[1]}, {dy[0]}, &staged) : 0;
        if (rc || staged || (rc = c.adj_add({e.args[1]}, mm(true, false), {dy[0], e.args[0]}))) return rc;
        std::unique_ptr<MatMulSpec> dx(new MatMulSpec(false, false, 1.f, 0));
        dx->lend = !one_launch(c.cell(dy[0]).ty, c.cell(e.args[1]).ty, 1);
        return c.adj_add({e.args[0]}, std::move(dx), {dy[0], e.args[1]});
    }
};

// ---------------------------------------------------------------------------
// RoPE (symplectic_embed src/librarium/llama.rs:463-465); cos/sin are const_ cells
// x is [S, H*Dh] (the reference's [1,S,H,Dh] flattened); the head count rides in the spec.
struct RopeBwdSpec : ThunkSpec {
    int64_t H;
    explicit RopeBwdSpec(int64_t h) : H(h) {}
    const char *name() const override { return "rope_bwd"; }
    int arity() const override { return 3; }                       // (dy, cos, sin) -> dx
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == F16 && a[0].shape.size() == 2 && a[0].shape[1] % H == 0,
                   "rope_bwd: dy f16 [S,H*Dh] expected");
        o = {a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        const auto &s = aty[0].shape;
        return cacti_hip_rope_bwd(s[0], H, s[1] / H, a[0], a[1], a[2], o[0], acc & 1, S(c));
    }
};

// The map on the query and the key of a layer in one launch: (q, k, cos, sin) -> (qr, kr), adjoint
// (dqr, dkr, cos, sin) -> (dq, dk); values as from two RopeSpec thunks.
struct Rope2BwdSpec : ThunkSpec {
    int64_t H;
    explicit Rope2BwdSpec(int64_t h) : H(h) {}
    const char *name() const override { return "rope2_bwd"; }
    int arity() const override { return 4; }
    int nout() const override { return 2; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == F16 && a[0].shape.size() == 2 && a[0].shape[1] % H == 0 && a[1] == a[0],
                   "rope2_bwd: two dy f16 [S,H*Dh] expected");
        o = {a[0], a[1]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        const auto &s = aty[0].shape;
        return cacti_hip_rope_bwd_pair(s[0], H, s[1] / H, a[0], a[1], a[2], a[3], o[0], acc & 1, o[1], (acc >> 1) & 1, S(c));
    }
};

struct Rope2Spec : ThunkSpec {
    int64_t H;
    explicit Rope2Spec(int64_t h) : H(h) {}
    const char *name() const override { return "rope2"; }
    int arity() const override { return 4; }
    int nout() const override { return 2; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == F16 && a[0].shape.size() == 2 && a[0].shape[1] % H == 0 && a[1] == a[0] &&
                       a[2].shape.size() == 2 && a[2].shape[0] >= a[0].shape[0] &&
                       a[2].shape[1] == a[0].shape[1] / H && a[2] == a[3],
                   "rope2: (q, k f16 [S,H*Dh], cos [S,Dh], sin [S,Dh]) expected");
        o = {a[0], a[1]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t, void *, size_t) const override
    {
        const auto &s = aty[0].shape;
        return cacti_hip_rope_fwd_pair(s[0], H, s[1] / H, a[0], a[1], a[2], a[3], o[0], o[1], S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        // one of the two without an adjoint: the single-tensor thunk for the other
        if (!dy[0] && !dy[1]) return 0;
        if (!dy[0] || !dy[1]) {
            const int k = dy[0] ? 0 : 1;
            return c.adj_add({e.args[k]}, std::unique_ptr<ThunkSpec>(new RopeBwdSpec(H)), {dy[k], e.args[2], e.args[3]});
        }
        return c.adj_add({e.args[0], e.args[1]}, std::unique_ptr<ThunkSpec>(new Rope2BwdSpec(H)),
                         {dy[0], dy[1], e.args[2], e.args[3]});
    }
};

struct RopeSpec : ThunkSpec {
    int64_t H;
    explicit RopeSpec(int64_t h) : H(h) {}
    const char *name() const override { return "rope"; }
    int arity() const override { return 3; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == F16 && a[0].shape.size() == 2 && a[0].shape[1] % H == 0 &&
                       a[1].shape.size() == 2 && a[1].shape[0] >= a[0].shape[0] &&
                       a[1].shape[1] == a[0].shape[1] / H && a[1] == a[2],
                   "rope: (x f16 [S,H*Dh], cos [S,Dh], sin [S,Dh]) expected");
        o = {a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t, void *, size_t) const override
    {
        const auto &s = aty[0].shape;
        return cacti_hip_rope_fwd(s[0], H, s[1] / H, a[0], a[1], a[2], o[0], S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        return c.adj_add({e.args[0]}, std::unique_ptr<ThunkSpec>(new RopeBwdSpec(H)),
                         {dy[0], e.args[1], e.args[2]});
    }
};

// ---------------------------------------------------------------------------
// causal softmax over scores (src/librarium/llama.rs:501-505)
struct CausalSoftmaxBwdSpec : ThunkSpec {
    int64_t H;
    explicit CausalSoftmaxBwdSpec(int64_t h) : H(h) {}
    const char *name() const override { return "causal_softmax_bwd"; }
    int arity() const override { return 2; }                       // (s16, dp16) -> ds16
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0] == a[1], "causal_softmax_bwd: shape mismatch");
        o = {a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        TY_REQUIRE(!(acc & 1), "causal_softmax_bwd: accumulate mode not staged on this path");
        return cacti_hip_causal_softmax_bwd(aty[0].shape[0], H, a[0], a[1], o[0], S(c));
    }
};

struct CausalSoftmaxSpec : ThunkSpec {
    int64_t H;
    explicit CausalSoftmaxSpec(int64_t h) : H(h) {}
    const char *name() const override { return "causal_softmax"; }
    int arity() const override { return 1; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == F16 && a[0].shape.size() == 2 && a[0].shape[1] == H * a[0].shape[0],
                   "causal_softmax: s16 f16 [S,H*S] expected");
        o = {a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t, void *, size_t) const override
    {
        return cacti_hip_causal_softmax_fwd(aty[0].shape[0], H, a[0], o[0], S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        return c.adj_add({e.args[0]}, std::unique_ptr<ThunkSpec>(new CausalSoftmaxBwdSpec(H)),
                         {e.args[0], dy[0]});
    }
};

// ---------------------------------------------------------------------------
// The attention block of a layer as one thunk: scores, cast, mask, softmax, cast and the product with
// v (src/librarium/llama.rs:501-507) with the rounding points of the separate thunks; the adjoint thunk
// stands for the adjoints of all of them.  q, k, v, o: [S, H*Dh]; stats: f32 [2*H*S].
struct AttentionBwdSpec : ThunkSpec {
    int64_t H;
    float alpha;
    AttentionBwdSpec(int64_t h, float a) : H(h), alpha(a) {}
    const char *name() const override { return "attention_bwd"; }
    int arity() const override { return 6; }                       // (q, k, v, dO, stats, o) -> dq, dk, dv
    int nout() const override { return 3; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0] == a[1] && a[0] == a[2] && a[0] == a[3] && a[0] == a[5] && a[0].shape.size() == 2 &&
                       a[4].dtype == F32,
                   "attention_bwd: (q, k, v, dO f16 [S,H*Dh], stats f32, o) expected");
        o = {a[0], a[0], a[0]};
        return 0;
    }
    size_t workspace(const std::vector<CellType> &a) const override { return cacti_hip_attention_bwd_workspace(a[0].shape[0], H); }
    size_t workspace_best(const std::vector<CellType> &a) const override
    {
        return cacti_hip_attention_bwd_workspace_used(a[0].shape[0], H, a[0].shape[1] / H, a[0].shape[1]);
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *ws, size_t wsb) const override
    {
        const auto &s = aty[0].shape;
        return cacti_hip_attention_bwd(s[0], H, s[1] / H, alpha, a[0], a[1], a[2], a[5], a[3], s[1], a[4], o[0],
                                       acc & 1, o[1], (acc >> 1) & 1, o[2], (acc >> 2) & 1, ws, wsb, S(c));
    }
};

struct AttentionSpec : ThunkSpec {
    int64_t H;
    float alpha;
    AttentionSpec(int64_t h, float a) : H(h), alpha(a) {}
    const char *name() const override { return "attention"; }
    int arity() const override { return 3; }                       // (q, k, v) -> o, stats
    int nout() const override { return 2; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == F16 && a[0] == a[1] && a[0] == a[2] && a[0].shape.size() == 2 &&
                       a[0].shape[1] % H == 0,
                   "attention: (q, k, v f16 [S,H*Dh]) expected");
        o = {a[0], CellType({(int64_t)(cacti_hip_attention_stats_bytes(a[0].shape[0], H) / sizeof(float))}, F32)};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        TY_REQUIRE(acc == 0, "attention: accumulate mode not staged on this path");
        const auto &s = aty[0].shape;
        return cacti_hip_attention_fwd(s[0], H, s[1] / H, alpha, a[0], a[1], a[2], s[1], o[0], o[1], S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        if (!dy[0]) return 0;
        return c.adj_add({e.args[0], e.args[1], e.args[2]},
                         std::unique_ptr<ThunkSpec>(new AttentionBwdSpec(H, alpha)),
                         {e.args[0], e.args[1], e.args[2], dy[0], e.outs[1], e.outs[0]});
    }
};

// ---------------------------------------------------------------------------
// SiLU gate (src/librarium/llama.rs:526-527)
struct SiluGateBwdSpec : ThunkSpec {
    const char *name() const override { return "silu_gate_bwd"; }
    int arity() const override { return 3; }                       // (g, u, dh) -> dg, du
    int nout() const override { return 2; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0] == a[1] && a[0] == a[2], "silu_gate_bwd: shape mismatch");
        o = {a[0], a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        return cacti_hip_silu_gate_bwd(aty[0].numel(), a[0], a[1], a[2], o[0], acc & 1, o[1],
                                       (acc >> 1) & 1, S(c));
    }
};

struct SiluGateSpec : ThunkSpec {
    const char *name() const override { return "silu_gate"; }
    int arity() const override { return 2; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0] == a[1] && a[0].dtype == F16, "silu_gate: equal f16 shapes expected");
        o = {a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t, void *, size_t) const override
    {
        return cacti_hip_silu_gate_fwd(aty[0].numel(), a[0], a[1], o[0], S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        return c.adj_add({e.args[0], e.args[1]}, std::unique_ptr<ThunkSpec>(new SiluGateBwdSpec()),
                         {e.args[0], e.args[1], dy[0]});
    }
};

// ---------------------------------------------------------------------------
// LM loss (src/librarium/llama.rs:541-546)
struct SoftmaxCeBwdSpec : ThunkSpec {
    const char *name() const override { return "softmax_ce_bwd"; }
    int arity() const override { return 3; }                       // (logit, tok, dloss) -> dlogit
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].shape.size() == 2 && a[2].dtype == F32 && a[2].numel() == a[0].shape[0],
                   "softmax_ce_bwd: (logit [N,V], tok, dloss f32 [N]) expected");
        o = {a[0]};
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t acc, void *, size_t) const override
    {
        return cacti_hip_softmax_ce_bwd(aty[0].shape[0], aty[0].shape[1], a[0], a[1], a[2], o[0],
                                        acc & 1, S(c));
    }
};

struct SoftmaxCeSpec : ThunkSpec {
    bool want_prob;
    explicit SoftmaxCeSpec(bool p) : want_prob(p) {}
    const char *name() const override { return "softmax_ce"; }
    int arity() const override { return 2; }
    int nout() const override { return want_prob ? 3 : 2; }
    int out_ty(const std::vector<CellType> &a, std::vector<CellType> &o) const override
    {
        TY_REQUIRE(a[0].dtype == F16 && a[0].shape.size() == 2 && a[1].dtype == U16 &&
                       a[1].numel() == a[0].shape[0],
                   "softmax_ce: (logit f16 [N,V], tok u16 [N]) expected");
        o = {CellType({a[0].shape[0]}, F32), CellType({a[0].shape[0]}, U16)};
        if (want_prob) o.push_back(CellType(a[0].shape, F32));
        return 0;
    }
    int run(Ctx &c, const std::vector<CellType> &aty, void *const *a, const std::vector<CellType> &,
            void *const *o, uint32_t, void *, size_t) const override
    {
        return cacti_hip_softmax_ce_fwd(aty[0].shape[0], aty[0].shape[1], a[0], a[1],
                                        want_prob ? o[2] : nullptr, o[0], o[1], c.status_ptr(), S(c));
    }
    int pop_adj(Ctx &c, const Entry &e, const std::vector<CellPtr> &dy) const override
    {
        if (!dy[0]) return 0;                    // only the loss output carries a gradient
        return c.adj_add({e.args[0]}, std::unique_ptr<ThunkSpec>(new SoftmaxCeBwdSpec()),
                         {e.args[0], e.args[1], dy[0]});
    }
};

}  // namespace

std::unique_ptr<ThunkSpec> make_embed() { return std::unique_ptr<ThunkSpec>(new EmbedSpec()); }
std::unique_ptr<ThunkSpec> make_row_sums(std::vector<CellType> ty) { return std::unique_ptr<ThunkSpec>(new RmsNormDwSpec(std::move(ty))); }
std::unique_ptr<ThunkSpec> make_rms_norm(float eps)
{
    return std::unique_ptr<ThunkSpec>(new RmsNormSpec(eps));
}
std::unique_ptr<ThunkSpec> make_matmul(bool ta, bool tb, float alpha)
{
    return std::unique_ptr<ThunkSpec>(new MatMulSpec(ta, tb, alpha, 0));
}
std::unique_ptr<ThunkSpec> make_linear(bool one) { return std::unique_ptr<ThunkSpec>(new LinearSpec(one)); }
std::unique_ptr<ThunkSpec> make_projections(int n, bool group_adjoints)
{
    return std::unique_ptr<ThunkSpec>(new ProjNSpec(n, group_adjoints));
}
std::unique_ptr<ThunkSpec> make_block_matmul(bool ta, bool tb, float alpha, int64_t H)
{
    return std::unique_ptr<ThunkSpec>(new MatMulSpec(ta, tb, alpha, H));
}
std::unique_ptr<ThunkSpec> make_causal_scores(float alpha, int64_t H)
{
    return std::unique_ptr<ThunkSpec>(new MatMulSpec(false, true, alpha, H, CAUSAL_OUT));
}
std::unique_ptr<ThunkSpec> make_causal_pv(int64_t H)
{
    return std::unique_ptr<ThunkSpec>(new MatMulSpec(false, false, 1.f, H, CAUSAL_A));
}
std::unique_ptr<ThunkSpec> make_rope(int64_t H) { return std::unique_ptr<ThunkSpec>(new RopeSpec(H)); }
std::unique_ptr<ThunkSpec> make_rope2(int64_t H) { return std::unique_ptr<ThunkSpec>(new Rope2Spec(H)); }
std::unique_ptr<ThunkSpec> make_causal_softmax(int64_t H)
{
    return std::unique_ptr<ThunkSpec>(new CausalSoftmaxSpec(H));
}
std::unique_ptr<ThunkSpec> make_attention(float alpha, int64_t H)
{
    return std::unique_ptr<ThunkSpec>(new AttentionSpec(H, alpha));
}
std::unique_ptr<ThunkSpec> make_add() { return std::unique_ptr<ThunkSpec>(new AddSpec()); }
std::unique_ptr<ThunkSpec> make_add_rms_norm(float eps)
{
    return std::unique_ptr<ThunkSpec>(new AddRmsNormSpec(eps));
}
std::unique_ptr<ThunkSpec> make_copy() { return std::unique_ptr<ThunkSpec>(new CopySpec()); }
std::unique_ptr<ThunkSpec> make_silu_gate()
{
    return std::unique_ptr<ThunkSpec>(new SiluGateSpec());
}
std::unique_ptr<ThunkSpec> make_softmax_ce(bool want_prob)
{
    return std::unique_ptr<ThunkSpec>(new SoftmaxCeSpec(want_prob));
}

}  // namespace cacti
