// Numerical-health digests over f16 tensors, integer-exact: the NaN count and the histogram of
// floor(log2 |x|) classes that the reference's training example takes of every parameter and
// gradient each cycle (NanCountFutThunkSpec, src/thunk/op.rs:273-349; AbsLog2Hist8FutThunkSpec,
// src/thunk/op.rs:351-441; used at examples/open_llama_3b_train.rs:409-424).
//
// Both stream the tensor once, 16 bytes per lane per step, and counting has to keep up with 6 TB/s: 8 elements per lane in
// some 40 clocks of its SIMD.  An LDS add per element, into the dozen adjacent bins that the values of a weight or gradient
// tensor fall into, did not (3.7 TB/s), nor did one per pair of elements (4.0).  So a lane counts in registers: 16 counters of
// four bits, for 16 neighbouring classes (Window), take 8 elements before they move to bytes, and those go to LDS once per 28
// pieces, summed over the wave.  Where a wave's 16 classes lie its first elements say (the largest, and one class more); pieces of 8
// elements with one beyond them, a zero among others or a NaN, one in 820 to 1130 of a normally distributed tensor (a wave has one
// in 13 to 18 of its steps), are counted in LDS, by pairs: the two exponent fields of a 32-bit word are one of 1024 bins, so there are half as many adds and
// they spread over a hundred addresses (four sets of bins, by lane & 3).  What an exponent field does not say, the
// subnormals' highest mantissa bit and the NaNs, is looked for in two halves at a time there and counted apart where there is
// any; zeros are the zero exponents that were not subnormal.  At the end of a workgroup the pairs are summed to exponents and
// each non-empty class is flushed with one 64-bit atomic.  Counts are integers: the order of the adds does not matter.
// 97 M elements in 12 tensors, with the launch that clears the counts: 47.3 -> 41.7 us (that launch and the reading alone: 34).
#include "common.h"

#include <algorithm>
#include <type_traits>

using namespace cacti;

namespace {

constexpr int kThreads = 256;
constexpr int kSets = 4;                   // sets of pair bins
constexpr int kSetPitch = 1024 + 16;       // their distance: the sets start in different banks

__device__ __forceinline__ int is_nan16(uint32_t u) { return (u & 0x7c00) == 0x7c00 && (u & 0x3ff) != 0; }

__global__ void __launch_bounds__(64) zero_i64_kernel(unsigned long long *p, int n)
{
    for (int i = blockIdx.x * 64 + threadIdx.x; i < n; i += gridDim.x * 64) p[i] = 0;
}

// one tensor of a launch: workgroups first_block .. first_block + blocks - 1 read it, sweep by sweep in turn (workgroup b
// takes sweeps b, b + blocks, ..: what the launch reads at a time is contiguous.  With a contiguous 128 KiB for each
// workgroup all of them walked the same addresses modulo 128 KiB, and so the same memory channels, at once: 3.4 TB/s);
// out[0..255] += histogram (HIST), out[HIST ? 256 : 0] += NaN count (NANS)
struct DigestSeg {
    const uint16_t *x;
    int64_t n;
    int32_t first_block, blocks;
    unsigned long long *out;
};
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kUnroll = 4;                 // 16-byte loads in flight per lane
constexpr int kSweep = kThreads * kUnroll; // 16-byte units a workgroup reads per step
inline int64_t seg_blocks(int64_t n, int64_t sweeps)
{
    const int64_t b = (n / 8 + sweeps * kSweep - 1) / (sweeps * kSweep);
    return b < 1 ? 1 : b;
}

// Sweeps per workgroup of a launch that reads `total`: `least` while that gives no more workgroups than four per CU, which
// the device holds all at once, then as many as four per CU leave each.  More workgroups put their zeroing and flushing behind
// one another, and their atomics on the same few words: 97 M elements with 8 / 12 / 16 sweeps each 46.6 / 41.7 / 42.0 us.
inline int64_t sweeps_each(int64_t total, int64_t least)
{
    const int64_t wgs = 4 * (int64_t)device_cus();
    return std::max(least, (total + wgs - 1) / wgs);
}
constexpr int kLeastSweeps = 8;            // when many tensors share a launch
inline int64_t sweeps_of(int64_t n) { return (n / 8 + kSweep - 1) / kSweep; }
// one tensor alone: 1 to 8 sweeps at least, growing once there are about 1536 workgroups
inline int64_t sweeps_alone(int64_t n)
{
    return sweeps_each(sweeps_of(n), std::min<int64_t>(8, std::max<int64_t>(1, (sweeps_of(n) + 1535) / 1536)));
}

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// Classes of the reference (src/thunk/op.rs:417-432): 255 for inf / nan, 0 for +-0, floor(log2 |x|) + 127 otherwise: exponent
// field + 112 for normal numbers, 103 + the index of the highest mantissa bit for subnormal ones.
struct Hist {
    uint32_t pair[kSets * kSetPitch];      // [set][exponent of the low half | exponent of the high half << 5]
    uint32_t expo[32], sub[10];
};

// subnormal halves and NaNs of a piece, one element at a time
template <bool NANS>
__device__ __forceinline__ void digest_rare(const uint32_t (&w)[4], Hist *h, uint32_t &nans)
{
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t x = w[i >> 1] >> (i & 1 ? 16 : 0) & 0x7fff;
        if (x - 1 < 0x3ff) atomicAdd(&h->sub[31 - __builtin_clz(x)], 1u);
        if (NANS) nans += x > 0x7c00;
    }
}

template <bool NANS>
__device__ __forceinline__ void digest_unit(const u32x4 v, uint32_t *pairs, Hist *h, uint32_t &nans)
{
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    u16x2 least = {0xffff, 0xffff}, most = {0, 0};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t x = w[i] & 0x7fff7fff, t = x >> 10 & 0x001f001f;
        atomicAdd(pairs + ((t | t >> 11) & 0x3ff), 1u);
        const u16x2 xv = __builtin_bit_cast(u16x2, x), one = {1, 1};
        most = __builtin_elementwise_max(most, xv);
        least = __builtin_elementwise_min(least, (u16x2)(xv - one));          // a zero wraps to the largest value
    }
    if (least.x < 0x3ff || least.y < 0x3ff || most.x > 0x7c00 || most.y > 0x7c00) digest_rare<NANS>(w, h, nans);
}

// The 16 classes that a wave counts in registers: numbers first .. first + 15 of 40 (0 .. 9 subnormal by their highest mantissa
// bit, 9 + the exponent field above), as f16 patterns lo .. hi.
struct Window {
    uint32_t lo, hi;                       // the pattern in both halves; lo > hi: no register counts
    int first;
};
__device__ __forceinline__ uint32_t least_of_class(int c) { return c < 10 ? 1u << c : (uint32_t)(c - 9) << 10; }
// largest: the largest |x| pattern of the wave's first elements
__device__ __forceinline__ Window window_for(uint32_t largest)
{
    const int e = min((int)(largest >> 10), 30), top = e ? e + 9 : largest ? 31 - __builtin_clz(largest) : 15;
    Window w;
    w.first = max(top - 14, 0);
    w.lo = least_of_class(w.first) * 0x10001u;
    w.hi = (least_of_class(min(w.first + 16, 40)) - 1) * 0x10001u;
    return w;
}

// A lane's counters: byte j of by[0], by[1] counts classes 2 j and 2 j + 8 modulo 16 of the f32 exponent, of by[2], by[3] the ones behind.
// At most 31 pieces of 8 fit in (28: kUnroll at a time) before they are flushed.
struct LaneCounts {
    uint32_t by[4], zeros;
};

template <bool NANS>
__device__ __forceinline__ void digest_piece(const u32x4 v, const Window &win, LaneCounts &c, uint32_t *pairs, Hist *h, uint32_t &nans)
{
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
    auto mag = [&](int i) __attribute__((always_inline)) { return __builtin_bit_cast(u16x2, w[i] & 0x7fff7fffu); };
    const u16x2 m0 = mag(0), m1 = mag(1), m2 = mag(2), m3 = mag(3);
    const u16x2 most = __builtin_elementwise_max(__builtin_elementwise_max(m0, m1), __builtin_elementwise_max(m2, m3));
    const u16x2 least = __builtin_elementwise_min(__builtin_elementwise_min(m0, m1), __builtin_elementwise_min(m2, m3));
    const uint32_t over = __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(most, __builtin_bit_cast(u16x2, win.hi))),
                   under = __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2, win.lo), least));
    if ((over | under) == 0) {
        // floor(log2 |x|) is the exponent of x as f32 (a subnormal f16 is a normal f32); its low four bits pick the counter
        uint64_t a = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const half2_t x = __builtin_bit_cast(half2_t, w[i]);
            a += 1ull << (__builtin_bit_cast(uint32_t, (float)x[0]) >> 21 & 0x3c);
            a += 1ull << (__builtin_bit_cast(uint32_t, (float)x[1]) >> 21 & 0x3c);
        }
        const uint32_t lo = (uint32_t)a, hi = (uint32_t)(a >> 32), m = 0x0f0f0f0fu;
        c.by[0] += lo & m;
        c.by[1] += hi & m;
        c.by[2] += lo >> 4 & m;
        c.by[3] += hi >> 4 & m;
    } else if (__builtin_bit_cast(uint32_t, most) == 0) {
        c.zeros += 8;                                       // (a tensor that is mostly zeros would add to one bin)
    } else {
        digest_unit<NANS>(v, pairs, h, nans);
    }
}

// the counters of a wave's lanes to LDS, and zeroed
__device__ __forceinline__ void flush_counts(const Window &win, LaneCounts &c, Hist *h, int lane)
{
    uint32_t mine = 0;
    auto sum = [](uint32_t a, uint32_t b) __attribute__((always_inline)) { return a + b; };
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int odd = 0; odd < 2; odd++) {
            // bytes odd and odd + 2, two sums of 64 x 255 at most
            const uint32_t s = wave_reduce(c.by[k] >> 8 * odd & 0x00ff00ffu, sum);
            const int n = 8 * (k & 1) + (k >> 1) + 2 * odd;
            mine = lane == n ? s & 0xffff : lane == n + 4 ? s >> 16 : mine;
        }
#pragma unroll
    for (int k = 0; k < 4; k++) c.by[k] = 0;
    const uint32_t zeros = wave_reduce(c.zeros, sum);
    c.zeros = 0;
    if (lane == 0 && zeros) atomicAdd(&h->expo[0], zeros);
    // lane n < 16: the class of the window whose f32 exponent (103 + its number) is n modulo 16
    const int cls = win.first + ((lane - 103 - win.first) & 15);
    if (lane < 16 && mine) {
        if (cls < 10) atomicAdd(&h->sub[cls], mine);
        atomicAdd(&h->expo[cls < 10 ? 0 : cls - 9], mine);
    }
}

// The tensors of a launch, in the kernel's arguments: a table in device memory is a copy in front of the launch.
constexpr int kSegsPerLaunch = 64;
struct DigestArgs {
    int nseg;
    DigestSeg seg[kSegsPerLaunch];         // by first_block
};

template <bool HIST, bool NANS>
__global__ void __launch_bounds__(kThreads)
digest_kernel(DigestArgs args)
{
    __shared__ typename std::conditional<HIST, Hist, int>::type hist_mem;
    Hist *const hist = reinterpret_cast<Hist *>(&hist_mem);
    const int lane = threadIdx.x & 63;
    if (HIST) {
        for (int i = threadIdx.x; i < (int)(sizeof(Hist) / 4); i += kThreads) reinterpret_cast<uint32_t *>(hist)[i] = 0;
    }
    int seg = 0;
    for (int hi = args.nseg - 1; seg < hi;) {                 // last segment starting at or before this block
        const int mid = (seg + hi + 1) >> 1;
        if (args.seg[mid].first_block <= (int)blockIdx.x) seg = mid;
        else hi = mid - 1;
    }
    const DigestSeg sg = args.seg[seg];
    if (HIST) __syncthreads();
    const int lb = (int)blockIdx.x - sg.first_block;
    uint32_t *pairs = hist->pair + (lane & (kSets - 1)) * kSetPitch;
    uint32_t nans = 0;
    const int64_t n8 = sg.n / 8;                                  // whole 16-byte units (x is 16-byte aligned)
    const u32x4 *xv = reinterpret_cast<const u32x4 *>(sg.x);
    auto nan_unit = [&](const u32x4 v) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int i = 0; i < 4; i++) nans += is_nan16(w[i] & 0xffff) + is_nan16(w[i] >> 16);
    };
    int64_t u = (int64_t)lb * kSweep;                             // the sweep's first unit
    const int64_t stride = (int64_t)sg.blocks * kSweep;
    u32x4 v[kUnroll], vn[kUnroll];
    auto load = [&](u32x4 (&d)[kUnroll], int64_t at) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kUnroll; j++) d[j] = __builtin_nontemporal_load(xv + at + j * kThreads + threadIdx.x);
    };
    Window win = {0x00010001u, 0u, 0};
    LaneCounts counts = {};
    int pieces = 0;                                               // in the lane's counters
    if (u + kSweep <= n8) {
        load(v, u);
        if (HIST) {
            uint32_t largest = 0;
#pragma unroll
            for (int j = 0; j < kUnroll; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) largest = max(largest, max(v[j][i] & 0x7fff, v[j][i] >> 16 & 0x7fff));
            win = window_for(wave_reduce(largest, [](uint32_t a, uint32_t b) __attribute__((always_inline)) { return max(a, b); }));
        }
    }
    for (; u + kSweep <= n8; u += stride) {
        load(vn, u + stride + kSweep <= n8 ? u + stride : u);     // the next sweep is on its way while this one is counted
        if (HIST && (pieces += kUnroll) > 31) {
            flush_counts(win, counts, hist, lane);
            pieces = kUnroll;
        }
#pragma unroll
        for (int j = 0; j < kUnroll; j++) {
            if (HIST) digest_piece<NANS>(v[j], win, counts, pairs, hist, nans);
            else nan_unit(v[j]);
        }
#pragma unroll
        for (int j = 0; j < kUnroll; j++) v[j] = vn[j];
    }
    if (HIST) flush_counts(win, counts, hist, lane);
    for (u += threadIdx.x; u < n8; u += kThreads) {               // the tensor's last, incomplete sweep
        const u32x4 t = xv[u];
        if (HIST) digest_unit<NANS>(t, pairs, hist, nans);
        else nan_unit(t);
    }
    // the last n % 8 elements: one lane each of the tensor's first workgroup
    if (lb == 0 && threadIdx.x < (int)(sg.n - n8 * 8)) {
        const uint32_t x = sg.x[n8 * 8 + threadIdx.x] & 0x7fff;
        if (HIST) {
            atomicAdd(&hist->expo[x >> 10], 1u);
            if (x - 1 < 0x3ff) atomicAdd(&hist->sub[31 - __builtin_clz(x)], 1u);
        }
        nans += x > 0x7c00;
    }
    if (HIST) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 1024 / kThreads; k++) {
            const int p = threadIdx.x + k * kThreads;
            uint32_t s = 0;
#pragma unroll
            for (int set = 0; set < kSets; set++) s += hist->pair[set * kSetPitch + p];
            if (s) {
                atomicAdd(&hist->expo[p & 31], s);
                atomicAdd(&hist->expo[p >> 5], s);
            }
        }
        __syncthreads();
        uint32_t s = 0;
        int bin = 0;
        if (threadIdx.x < 32) {
            s = hist->expo[threadIdx.x];
            bin = threadIdx.x == 31 ? 255 : (int)threadIdx.x + 112;
            if (threadIdx.x == 0) {
                bin = 0;
                for (int i = 0; i < 10; i++) s -= hist->sub[i];
            }
        } else if (threadIdx.x < 42) {
            s = hist->sub[threadIdx.x - 32];
            bin = 103 + (int)threadIdx.x - 32;
        }
        if (s) atomicAdd(&sg.out[bin], (unsigned long long)s);
    }
    if (NANS) {
        // wave sum of the lane counts, then one atomic per wave
        for (int off = 32; off > 0; off >>= 1) nans += __shfl_down(nans, off, 64);
        if (lane == 0 && nans) atomicAdd(sg.out + (HIST ? 256 : 0), (unsigned long long)nans);
    }
}

template <bool HIST, bool NANS>
int run(int64_t n, const void *x, void *out, hipStream_t st)
{
    hipLaunchKernelGGL(zero_i64_kernel, dim3(1), dim3(64), 0, st, (unsigned long long *)out,
                       (HIST ? 256 : 0) + (NANS ? 1 : 0));
    if (n > 0) {
        DigestArgs args;
        args.nseg = 1;
        const int64_t blocks = seg_blocks(n, sweeps_alone(n));
        CACTI_REQUIRE(blocks < (int64_t)1 << 31, CACTI_E_INVALID, "digest: tensor too large for one launch");
        args.seg[0] = {(const uint16_t *)x, n, 0, (int32_t)blocks, (unsigned long long *)out};
        hipLaunchKernelGGL((digest_kernel<HIST, NANS>), dim3((unsigned)blocks), dim3(kThreads), 0, st, args);
    }
    return launch_status(HIST ? "abs_log2_hist8" : "nan_count");
}

}  // namespace

namespace cacti {
int digest_batch_f16(int count, const void *const *xs, const int64_t *ns, void *out, hipStream_t st);
}  // namespace cacti

CACTI_API int cacti_hip_nan_count_f16(int64_t n, const void *x, void *count_i64, void *stream)
{
    CACTI_REQUIRE(n >= 0 && count_i64 && (x || n == 0), CACTI_E_INVALID, "nan_count: null pointer or negative size");
    CACTI_REQUIRE(aligned(x, 16) && aligned(count_i64, 8), CACTI_E_INVALID,
                  "nan_count: x must be 16-byte aligned, the count 8-byte aligned");
    return run<false, true>(n, x, count_i64, (hipStream_t)stream);
}

CACTI_API int cacti_hip_abs_log2_hist8_f16(int64_t n, const void *x, void *hist_i64_256, void *stream)
{
    CACTI_REQUIRE(n >= 0 && hist_i64_256 && (x || n == 0), CACTI_E_INVALID,
                  "abs_log2_hist8: null pointer or negative size");
    CACTI_REQUIRE(aligned(x, 16) && aligned(hist_i64_256, 8), CACTI_E_INVALID,
                  "abs_log2_hist8: x must be 16-byte aligned, the histogram 8-byte aligned");
    return run<true, false>(n, x, hist_i64_256, (hipStream_t)stream);
}

CACTI_API size_t cacti_hip_digests_scratch_bytes(int) { return 0; }

CACTI_API int cacti_hip_digests_f16_batch(int count, const void *const *xs, const int64_t *ns, void *out_i64,
                                          void *, void *stream)
{
    CACTI_REQUIRE(count >= 0, CACTI_E_INVALID, "digests_batch: negative count");
    if (count == 0) return 0;
    CACTI_REQUIRE(xs && ns && out_i64 && aligned(out_i64, 8), CACTI_E_INVALID,
                  "digests_batch: null or misaligned argument");
    return cacti::digest_batch_f16(count, xs, ns, out_i64, (hipStream_t)stream);
}

namespace cacti {

// Both digests of `count` tensors, up to kSegsPerLaunch of them in a launch: out[257 * i + 0..255] = histogram and
// out[257 * i + 256] = NaN count of tensor i.  xs[i] 16-byte aligned, ns[i] >= 0.
int digest_batch_f16(int count, const void *const *xs, const int64_t *ns, void *out, hipStream_t st)
{
    if (count <= 0) return 0;
    for (int i = 0; i < count; i++)
        CACTI_REQUIRE(ns[i] >= 0 && ns[i] < (int64_t)1 << 44 && (xs[i] || ns[i] == 0) && aligned(xs[i], 16), CACTI_E_INVALID,
                      "digest_batch: tensor %d: null, bad size or not 16-byte aligned", i);
    hipLaunchKernelGGL(zero_i64_kernel, dim3(64), dim3(64), 0, st, (unsigned long long *)out, count * 257);
    for (int i0 = 0; i0 < count; i0 += kSegsPerLaunch) {
        DigestArgs args;
        args.nseg = count - i0 < kSegsPerLaunch ? count - i0 : kSegsPerLaunch;
        int64_t blocks = 0, total = 0;
        for (int i = 0; i < args.nseg; i++) total += sweeps_of(ns[i0 + i]);
        const int64_t each = sweeps_each(total, kLeastSweeps);
        for (int i = 0; i < args.nseg; i++) {
            const int64_t nb = seg_blocks(ns[i0 + i], each);
            CACTI_REQUIRE(blocks + nb < (int64_t)1 << 31, CACTI_E_INVALID, "digest_batch: too many workgroups");
            args.seg[i] = {(const uint16_t *)xs[i0 + i], ns[i0 + i], (int32_t)blocks, (int32_t)nb, (unsigned long long *)out + (size_t)(i0 + i) * 257};
            blocks += nb;
        }
        hipLaunchKernelGGL((digest_kernel<true, true>), dim3((unsigned)blocks), dim3(kThreads), 0, st, args);
    }
    return launch_status("digest_batch");
}

}  // namespace cacti
