// RMSNorm forward and adjoint, one 64-lane wavefront per row.
//
// A row (D halves) lives in registers as CH 16-byte chunks per lane, loaded once
// from HBM; the two row reductions (sum x^2, sum dt*x) are DPP wave reductions, so
// a row needs no barrier.  The adjoint keeps the reference's rounding schedule:
//   du = f32(dy); t = f32(x)/r; dw += f32(f16(du t)); dt = du f32(w);
//   c1 = f16(dt / r); dr = -sum(dt x)/r^2; ds = dr/(r+r); dsq = ds/D;
//   c2 = f16(dsq (x+x)); dx = f16(f16(dx_old + c1) + c2)   (or f16(c1 + c2))
// (rms_norm closure src/librarium/llama.rs:442-451 and its adjoint chain).
#include "rmsnorm.h"
#include "softmax_math.h"

using namespace cacti;

namespace {

constexpr int kWaves = 8;                 // rows per block
constexpr int kThreads = kWaves * 64;

// x2 != nullptr: the row is first formed as x = f16(x + x2) (the residual add in front of the
// norm, one thunk boundary) and also written to `sum`
template <int CH>
__global__ void __launch_bounds__(kThreads)
rms_norm_fwd_kernel(int64_t N, int D, const half_t *__restrict__ x, const half_t *__restrict__ x2,
                    const half_t *__restrict__ w, float eps, half_t *__restrict__ sum,
                    half_t *__restrict__ y)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t n = (int64_t)blockIdx.x * kWaves + wid;
    if (n >= N) return;
    const int nchunk = D / 8;
    const half_t *xr = x + n * D;
    // All loads of the row are issued first and unconditionally (chunks past the row re-read its
    // last chunk): a load inside `if (ch < nchunk)` is waited for at the end of that branch, which
    // makes the CH loads of a lane CH round trips.
    h8 xv[CH], bv[CH], wv[CH];
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int ch = min(c * 64 + lane, nchunk - 1);
        xv[c] = ld8(xr + ch * 8);
        if (x2) bv[c] = ld8(x2 + n * D + ch * 8);         // uniform over the launch
        wv[c] = ld8(w + ch * 8);
    }
    // the squares of f16 values are exact in fp32; summed in fp64 the row sum is the exactly rounded
    // one, whatever the order, so r is the reference's r and not one of its neighbours
    double ss = 0.0;
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int ch = c * 64 + lane;
        if (ch < nchunk) {
            if (x2) {
#pragma unroll
                for (int i = 0; i < 8; i++) xv[c].v[i] = f2h(h2f(xv[c].v[i]) + h2f(bv[c].v[i]));
                st8(sum + n * D + ch * 8, xv[c]);
            }
#pragma unroll
            for (int i = 0; i < 8; i++) {
                float f = h2f(xv[c].v[i]);
                ss += (double)(f * f);
            }
        }
    }
    ss = wave_sum_f64(ss);
    // t = x / r as the reference divides: a reciprocal and one residual correction give the
    // correctly rounded quotient (x * (1/r) alone is an ulp off for a quarter of the elements, and
    // in a chain of f16-rounded products that ulp grows like any other change of rounding)
    const RowDivide div(sqrtf((float)ss / (float)D + eps));
    half_t *yr = y + n * D;
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int ch = c * 64 + lane;
        if (ch < nchunk) {
            h8 o;
#pragma unroll
            for (int i = 0; i < 8; i++) o.v[i] = f2h(h2f(wv[c].v[i]) * div(h2f(xv[c].v[i])));
            st8(yr + ch * 8, o);
        }
    }
}

// Some 25 vector instructions per element (the correctly rounded quotients, the fp64 sums), which are what it takes: 2048 x 3200
// 15.0 -> 14.0 us with that, two waves to a row 15.6.  f16 values that only meet f16 values again stay f16: their sum rounded to f16 is v_add_f16
// (24 bits of an fp32 sum rounded to 11 lose nothing: 24 >= 2 * 11 + 2).
template <int CH>
__global__ void __launch_bounds__(kThreads)
rms_norm_bwd_kernel(int64_t N, int D, const half_t *__restrict__ x, const half_t *__restrict__ w,
                    float eps, const half_t *__restrict__ dy, half_t *dx, int dx_acc,
                    float *__restrict__ dw_part)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    half_t *sdw = reinterpret_cast<half_t *>(smem_raw);   // [kWaves][D] f16(du t)
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t n = (int64_t)blockIdx.x * kWaves + wid;
    const int nchunk = D / 8;
    const bool live = n < N;

    h8 dwp[CH];
#pragma unroll
    for (int c = 0; c < CH; c++)
#pragma unroll
        for (int i = 0; i < 8; i++) dwp[c].v[i] = 0;

    if (live) {
        const half_t *xr = x + n * D, *gr = dy + n * D;
        // every load of the row up front and unconditional (see the forward kernel), but for dx of rows beyond 8 chunks: with it a
        // lane spills 108 registers instead of 56 (2048 rows of 4608 43.0 us, 31.6 so; of 6144 55.3, 41.6; of 8192 95, 80;
        // accumulating 44.1, 34.6)
        half_t *or_ = dx + n * D;
        // without accumulation the fourth stream re-reads dy (a cache hit) instead of dx
        const half_t *oldr = dx_acc ? or_ : gr;
        constexpr bool EARLY = CH <= 8;
        h8 xv[CH], gv[CH], wv[CH], old[EARLY ? CH : 1];      // old: used only when dx accumulates
        double ss = 0.0;
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int ch = min(c * 64 + lane, nchunk - 1);
            xv[c] = ld8(xr + ch * 8);
            gv[c] = ld8(gr + ch * 8);
            wv[c] = ld8(w + ch * 8);
            if constexpr (EARLY) old[c] = ld8(oldr + ch * 8);
        }
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int ch = c * 64 + lane;
            if (ch < nchunk) {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    float f = h2f(xv[c].v[i]);
                    ss += (double)(f * f);
                }
            }
        }
        ss = wave_sum_f64(ss);                    // as in the forward kernel: the same r, bit for bit
        const float r = sqrtf((float)ss / (float)D + eps);
        const RowDivide div(r), div2(r * r);      // correctly rounded x / r, dt / r and (dt x) / r^2
        double sdx = 0.0;
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int ch = c * 64 + lane;
            if (ch < nchunk) {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    float xf = h2f(xv[c].v[i]), du = h2f(gv[c].v[i]);
                    float t = div(xf);
                    dwp[c].v[i] = f2h(du * t);
                    float dt = du * h2f(wv[c].v[i]);
                    sdx += (double)div2(dt * xf);       // the reference's per-element term of dr
                    gv[c].v[i] = f2h(div(dt));          // c1, kept in place of dy
                    // dt is needed no further: c2 depends only on the row sum
                }
            }
        }
        sdx = wave_sum_f64(sdx);
        const float dr = -(float)sdx;
        const float ds = dr / (r + r);
        const float dsq = ds / (float)D;
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int ch = c * 64 + lane;
            if (ch < nchunk) {
                h8 o;
                if constexpr (!EARLY) {
                    if (dx_acc) old[0] = ld8(or_ + ch * 8);
                }
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float xf = h2f(xv[c].v[i]);
                    const half_t c2 = f2h(dsq * (xf + xf)), c1 = gv[c].v[i];
                    o.v[i] = (dx_acc ? old[EARLY ? c : 0].v[i] + c1 : c1) + c2;
                }
                st8(or_ + ch * 8, o);
            }
        }
    }

    // block partial of dw: every wave stores its row at once, the columns are summed in the rows' order after one barrier
#pragma unroll
    for (int c = 0; c < CH; c++) {
        const int ch = c * 64 + lane;
        if (ch < nchunk) st8(sdw + wid * D + ch * 8, dwp[c]);
    }
    __syncthreads();
    float *dst = dw_part + (int64_t)blockIdx.x * D;
    for (int i = threadIdx.x * 8; i < D; i += blockDim.x * 8) {
        float a[8];
#pragma unroll
        for (int wv = 0; wv < kWaves; wv++) {
            const h8 r = ld8(sdw + wv * D + i);
#pragma unroll
            for (int k = 0; k < 8; k++) a[k] = wv ? a[k] + h2f(r.v[k]) : h2f(r.v[k]);
        }
        *reinterpret_cast<float4_t *>(dst + i) = float4_t{a[0], a[1], a[2], a[3]};
        *reinterpret_cast<float4_t *>(dst + i + 4) = float4_t{a[4], a[5], a[6], a[7]};
    }
}

// dw[d] (+)= f16(sum over block partials): a block owns 32 columns (8 lanes x float4) and
// splits the partial rows over 32 slices, so D / 32 blocks share the read of the partials.  A lane's rows, up to 8 of them, are
// requested together, as the launch is a chain of latencies (256 rows of 3200 4.59 -> 4.25 us, 98 of 2048 4.4 either way; norms,
// rotation and gate of 2048 rows in both directions 98.5 -> 97.0).
constexpr int kFinCols = 32, kFinSlices = 32, kFinRows = 8;
// The weights' gradients that a launch sums, one to a row of its grid: a training cycle's norms together, as each sum alone is all
// latency (two micro-batches of 611 positions, 4 layers of 1024: 18 launches of 4.25 us -> 2 of 4.0; 128 positions, 2 layers of
// 256: 5 of 2.5 -> 1 of 2.8; runs of the whole cycles differ by more than that).
struct DwSums {
    const float *part[kRmsNormDwSums];
    half_t *dw[kRmsNormDwSums];
    uint32_t acc;                              // bit i: dw[i] is added to
};
__global__ void __launch_bounds__(kFinCols / 4 * kFinSlices)
rms_norm_dw_finalize_kernel(int G, int D, DwSums p)
{
    const float *__restrict__ part = p.part[blockIdx.y];
    half_t *dw = p.dw[blockIdx.y];
    const bool acc = p.acc >> blockIdx.y & 1;
    __shared__ float red[kFinSlices][kFinCols];
    const int cg = threadIdx.x & (kFinCols / 4 - 1), slice = threadIdx.x / (kFinCols / 4);
    const int col = blockIdx.x * kFinCols + cg * 4;            // D % 8 == 0: a float4 is whole
    float4_t a = {0.f, 0.f, 0.f, 0.f};
    if (col < D)
        for (int g = slice; g < G; g += kFinSlices * kFinRows) {
            float4_t v[kFinRows];
#pragma unroll
            for (int j = 0; j < kFinRows; j++)
                v[j] = *reinterpret_cast<const float4_t *>(part + (int64_t)min(g + j * kFinSlices, G - 1) * D + col);
#pragma unroll
            for (int j = 0; j < kFinRows; j++)
                if (g + j * kFinSlices < G) a += v[j];
        }
#pragma unroll
    for (int i = 0; i < 4; i++) red[slice][cg * 4 + i] = a[i];
    __syncthreads();
    const int c = blockIdx.x * kFinCols + threadIdx.x;
    if (threadIdx.x < kFinCols && c < D) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < kFinSlices; i++) s += red[i][threadIdx.x];
        dw[c] = acc ? f2h(h2f(dw[c]) + rnd16(s)) : f2h(s);
    }
}

inline int ch_for(int64_t D) { return (int)((D / 8 + 63) / 64); }

template <int CH>
void launch_fwd(int64_t N, int D, const half_t *x, const half_t *x2, const half_t *w, float eps,
                half_t *sum, half_t *y, hipStream_t st)
{
    hipLaunchKernelGGL(rms_norm_fwd_kernel<CH>, dim3((unsigned)((N + kWaves - 1) / kWaves)),
                       dim3(kThreads), 0, st, N, D, x, x2, w, eps, sum, y);
}
template <int CH>
void launch_bwd(int64_t N, int D, const half_t *x, const half_t *w, float eps, const half_t *dy,
                half_t *dx, int dx_acc, float *part, hipStream_t st)
{
    const size_t smem = (size_t)kWaves * D * sizeof(half_t);      // 128 KB for the longest row
    auto kern = rms_norm_bwd_kernel<CH>;
    static DeviceOnce attr_set;                   // one per instantiation
    if (!attr_set.fresh()) {
        (void)hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  128 * 1024);
        attr_set.mark();
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)((N + kWaves - 1) / kWaves)), dim3(kThreads), smem, st,
                       N, D, x, w, eps, dy, dx, dx_acc, part);
}

}  // namespace

#define CACTI_DISPATCH_CH(ch, CALL)                 \
    switch (ch) {                                   \
        case 1: { constexpr int CH = 1; CALL; } break;   \
        case 2: { constexpr int CH = 2; CALL; } break;   \
        case 3: case 4: { constexpr int CH = 4; CALL; } break;   \
        case 5: case 6: case 7: { constexpr int CH = 7; CALL; } break;   \
        case 8: { constexpr int CH = 8; CALL; } break;   \
        case 9: case 10: case 11: case 12: { constexpr int CH = 12; CALL; } break; \
        default: { constexpr int CH = 16; CALL; } break; \
    }

CACTI_API int cacti_hip_rms_norm_fwd(int64_t N, int64_t D, const void *x, const void *w, float eps,
                                     void *y, void *stream)
{
    CACTI_REQUIRE(N > 0 && D > 0 && x && w && y, CACTI_E_INVALID,
                  "rms_norm_fwd: null pointer or empty shape");
    CACTI_REQUIRE(D % 8 == 0 && D <= 8192, CACTI_E_NOTIMPL,
                  "rms_norm_fwd: need D %% 8 == 0 and D <= 8192 (D=%lld)", (long long)D);
    CACTI_REQUIRE(aligned(x, 16) && aligned(w, 16) && aligned(y, 16), CACTI_E_INVALID,
                  "rms_norm_fwd: tensors must be 16-byte aligned");
    CACTI_DISPATCH_CH(ch_for(D), launch_fwd<CH>(N, (int)D, (const half_t *)x, nullptr, (const half_t *)w,
                                                eps, nullptr, (half_t *)y, (hipStream_t)stream));
    return launch_status("rms_norm_fwd");
}

CACTI_API int cacti_hip_add_rms_norm_fwd(int64_t N, int64_t D, const void *a, const void *b, const void *w,
                                         float eps, void *sum, void *y, void *stream)
{
    CACTI_REQUIRE(N > 0 && D > 0 && a && b && w && sum && y, CACTI_E_INVALID,
                  "add_rms_norm_fwd: null pointer or empty shape");
    CACTI_REQUIRE(D % 8 == 0 && D <= 8192, CACTI_E_NOTIMPL,
                  "add_rms_norm_fwd: need D %% 8 == 0 and D <= 8192 (D=%lld)", (long long)D);
    CACTI_REQUIRE(aligned(a, 16) && aligned(b, 16) && aligned(w, 16) && aligned(sum, 16) && aligned(y, 16),
                  CACTI_E_INVALID, "add_rms_norm_fwd: tensors must be 16-byte aligned");
    CACTI_DISPATCH_CH(ch_for(D), launch_fwd<CH>(N, (int)D, (const half_t *)a, (const half_t *)b,
                                                (const half_t *)w, eps, (half_t *)sum, (half_t *)y,
                                                (hipStream_t)stream));
    return launch_status("add_rms_norm_fwd");
}

CACTI_API size_t cacti_hip_rms_norm_bwd_workspace(int64_t N, int64_t D)
{
    if (N <= 0 || D <= 0) return 0;
    return (size_t)((N + kWaves - 1) / kWaves) * (size_t)D * sizeof(float);
}

namespace cacti {
int rms_norm_dw_sums(int n, int64_t G, int64_t D, const void *const *part, void *const *dw, uint32_t acc, hipStream_t st)
{
    CACTI_REQUIRE(n > 0 && n <= kRmsNormDwSums, CACTI_E_INVALID, "rms_norm_dw: %d sums", n);
    DwSums p = {};
    for (int i = 0; i < n; i++) {
        p.part[i] = (const float *)part[i];
        p.dw[i] = (half_t *)dw[i];
    }
    p.acc = acc;
    hipLaunchKernelGGL(rms_norm_dw_finalize_kernel, dim3((unsigned)((D + kFinCols - 1) / kFinCols), (unsigned)n),
                       dim3(kFinCols / 4 * kFinSlices), 0, st, (int)G, (int)D, p);
    return launch_status("rms_norm_dw_finalize");
}
}  // namespace cacti

static int rms_norm_bwd(int64_t N, int64_t D, const void *x, const void *w, float eps, const void *dy, void *dx, int dx_acc, void *dw,
                        int dw_acc, void *workspace, size_t workspace_bytes, void *stream)
{
    CACTI_REQUIRE(N > 0 && D > 0 && x && w && dy && dx && workspace, CACTI_E_INVALID,
                  "rms_norm_bwd: null pointer or empty shape");
    CACTI_REQUIRE(D % 8 == 0 && D <= 8192, CACTI_E_NOTIMPL,
                  "rms_norm_bwd: need D %% 8 == 0 and D <= 8192 (D=%lld)", (long long)D);
    CACTI_REQUIRE(aligned(x, 16) && aligned(w, 16) && aligned(dy, 16) && aligned(dx, 16) &&
                      aligned(workspace, 16),
                  CACTI_E_INVALID, "rms_norm_bwd: tensors must be 16-byte aligned");
    CACTI_REQUIRE(workspace_bytes >= cacti_hip_rms_norm_bwd_workspace(N, D), CACTI_E_INVALID,
                  "rms_norm_bwd: workspace of %zu bytes is smaller than the %zu needed",
                  workspace_bytes, cacti_hip_rms_norm_bwd_workspace(N, D));
    hipStream_t st = (hipStream_t)stream;
    CACTI_DISPATCH_CH(ch_for(D),
                      launch_bwd<CH>(N, (int)D, (const half_t *)x, (const half_t *)w, eps,
                                     (const half_t *)dy, (half_t *)dx, dx_acc, (float *)workspace,
                                     st));
    const int rc = launch_status("rms_norm_bwd");
    return rc || !dw ? rc : rms_norm_dw_sums(1, (N + kWaves - 1) / kWaves, D, (const void *const *)&workspace, &dw, dw_acc ? 1 : 0, st);
}

CACTI_API int cacti_hip_rms_norm_bwd(int64_t N, int64_t D, const void *x, const void *w, float eps,
                                     const void *dy, void *dx, int dx_acc, void *dw, int dw_acc,
                                     void *workspace, size_t workspace_bytes, void *stream)
{
    CACTI_REQUIRE(dw, CACTI_E_INVALID, "rms_norm_bwd: null pointer or empty shape");
    return rms_norm_bwd(N, D, x, w, eps, dy, dx, dx_acc, dw, dw_acc, workspace, workspace_bytes, stream);
}

namespace cacti {
int rms_norm_bwd_parts(int64_t N, int64_t D, const void *x, const void *w, float eps, const void *dy, void *dx, int dx_acc, void *part,
                       size_t part_bytes, hipStream_t st)
{
    return rms_norm_bwd(N, D, x, w, eps, dy, dx, dx_acc, nullptr, 0, part, part_bytes, st);
}
}  // namespace cacti

// ---- the same adjoint for callers that cannot allocate ----------------------------------------
// The fp32 dw partial rows go to a file-scope device array instead of a caller workspace.  The
// array's name is only a host-side stand-in: its device address is looked up once per device and
// that pointer, never the name, is what reaches the kernels.
namespace {
constexpr size_t kStaticScratchBytes = 8u << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
constexpr int kMaxDevices = 64;
void *g_scratch_ptr[kMaxDevices];          // per device, nullptr until first use on that device
unsigned g_scratch_epoch[kMaxDevices];     // the module epoch each address was taken in
}  // namespace

CACTI_API size_t cacti_hip_rms_norm_bwd_static_max_bytes(void) { return kStaticScratchBytes; }

CACTI_API int cacti_hip_rms_norm_bwd_static(int64_t N, int64_t D, const void *x, const void *w, float eps,
                                            const void *dy, void *dx, int dx_acc, void *dw, int dw_acc,
                                            void *stream)
{
    const size_t need = cacti_hip_rms_norm_bwd_workspace(N, D);
    CACTI_REQUIRE(N > 0 && D > 0 && need <= kStaticScratchBytes, CACTI_E_INVALID,
                  "rms_norm_bwd_static: N=%lld, D=%lld needs %zu bytes of scratch, the built-in buffer "
                  "holds %zu; use cacti_hip_rms_norm_bwd with a workspace",
                  (long long)N, (long long)D, need, kStaticScratchBytes);
    int dev = -1;
    CACTI_HIP(hipGetDevice(&dev));
    CACTI_REQUIRE(dev >= 0 && dev < kMaxDevices, CACTI_E_NOTIMPL,
                  "rms_norm_bwd_static: device %d is beyond the %d this entry point keeps a buffer for",
                  dev, kMaxDevices);
    if (!g_scratch_ptr[dev] || g_scratch_epoch[dev] != module_epoch()) {   // first use, or the modules were reloaded
        void *p = nullptr;
        CACTI_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        CACTI_REQUIRE(p != nullptr, CACTI_E_STATE, "rms_norm_bwd_static: no device address for the scratch array");
        g_scratch_ptr[dev] = p;
        g_scratch_epoch[dev] = module_epoch();
    }
    return cacti_hip_rms_norm_bwd(N, D, x, w, eps, dy, dx, dx_acc, dw, dw_acc, g_scratch_ptr[dev],
                                  kStaticScratchBytes, stream);
}
