// Attention of one to four new positions over the key / value cache (decoding): the chain
//   block_matmul_scale(q, k_cache^T, 1/sqrt(Dh)) -> f32 -> row-causal mask -> softmax -> f16
//   -> block_matmul(., v_cache)                      src/librarium/llama.rs:895-915
// with the reference's rounding points (scores and probabilities are f16 values, both products
// accumulate in fp32 and round once), but for probabilities over many positions, which stay f32.
//
// A single query row per head is a few hundred KB of cache and hardly any arithmetic: what it costs is launches and
// round trips to memory.  Up to some hundred positions a workgroup takes a head and a piece of its dimension (8 to 32 columns), over
// all positions, and every piece's workgroup forms the head's scores itself, K coming out of L2 for all but the first.
//
// Beyond, a workgroup takes 64, 128 or 256 positions of a head, and the last one of the head puts the parts together: up to 16
// of them, which a lane requests at once (16 heads of 128, 960 / 1200 positions with 64 each 5.8 / 7.6 us, with 128 6.4 / 6.8).
// The parts and the counter that tells the last one go past the L2s (store_shared), since a device-wide fence inside a launch costs
// 40 us on this chip; the counters have a cache line each (side by side they cost 2 to 4 us) and are cleared by the launch in front.
// Before there were parts, the scores were a launch of their own and every piece's workgroup read them all: 16 heads of 128,
// 600 / 960 / 1540 / 4000 / 8192 positions, without the gap between the launches 6.9 / 7.4 / 8.5 / 14.4 / 25.8 -> 5.5 / 5.8 /
// 7.6 / 11.1 / 17.1 us; 32 heads of 100 7.8 / 8.7 / 11.9 / 21.2 / 41.5 -> 6.8 / 7.8 / 9.9 / 16.4 / 30.1; four rows of 16 x 128
// 11.2 / 12.2 / 14.4 / 22.9 / 40.9 -> 9.0 / 9.6 / 11.8 / 17.2 / 26.1.  A prompt of 1531 and 16 tokens, 4 layers of 2048: 3752 -> 3676.
// Against 64 bits the result is no further off (1540 positions of 16 x 128 5.4e-4 -> 5.0e-4, 2000 of 32 x 100 5.7e-4 -> 5.4e-4).
//
// In the scores eight lanes share a position, each with 8-byte pieces of the head (a head starts on a multiple of 8
// bytes), 64 contiguous bytes per access; in the product with V it is LP lanes with a piece each.  (The head is the fast
// index of the grid: where their number is a multiple of 8, all workgroups of a head are on one XCD and share a row's
// bytes in its L2.)  Four positions per lane are in flight together, all of a part's; the first V pieces are requested once the
// scores' own loads are, which would otherwise be returned behind them, and arrive during the softmax.  Loads are unconditional
// with clamped indices: a load inside a branch is waited for at the end of the branch.
#include "common.h"
#include "gemm_internal.h"
#include "softmax_math.h"

#include <algorithm>

using namespace cacti;

namespace {

constexpr int kThreads = 256;              // of a launch in parts; one workgroup of all positions has kThreads or kWide
constexpr int kWide = 512;
constexpr int kStep = 4;                   // positions of a lane in flight
constexpr int kWordPitch = kClearPitch;    // words from a head's counter to the next
constexpr int kJoin = 16;                  // parts a lane of its last workgroup requests together
// Up to here kThreads lanes, eight to a position, own scores: one step over the positions, which more lanes cannot make
// shorter (70 positions, 32 heads of 100: 4.6 against 4.9 us; 300 positions 6.8 against 6.5).
constexpr int kNarrow = 128;
// Up to here kWide lanes, four to a position, a workgroup of all positions; beyond, parts of them.  Where a launch in front has cleared
// the counters, the parts are one launch (us, all positions against parts): 16 heads of 128, 250 / 400 / 480 positions 5.1 / 6.0 /
// 6.0 against 5.1 / 5.3 / 5.3, 32 heads of 100 5.0 / 6.5 / 6.6 against 5.2 / 5.5 / 5.8, four rows of 16 x 128 8.4 / 10.4 against
// 8.3 / 8.8; heads to 64, which have half of the keys' bytes to read, 32 of them 4.4 / 4.9 / 4.9 against 4.7 / 4.7 / 4.8.
constexpr int kOwnScoresCleared = 256, kOwnScoresShortCleared = 384;
// Where none has, they are two (600 / 960 positions, 16 heads of 128 6.6 / 6.8 us and the gap between them, 32 of 64 5.5 / 6.2),
// against a workgroup of all of 480 positions 6.0 and, of heads to 64, of 960 6.4.
constexpr int kOwnScores = 480, kOwnScoresShort = 960;
constexpr int kMaxCols = 8192;

struct __attribute__((aligned(8))) h4 {
    half_t v[4];
};

__device__ __forceinline__ float dot4(const h4 &a, const h4 &b, float acc)
{
    const half2_t a0 = {a.v[0], a.v[1]}, b0 = {b.v[0], b.v[1]}, a1 = {a.v[2], a.v[3]}, b1 = {b.v[2], b.v[3]};
    return __builtin_amdgcn_fdot2(a1, b1, __builtin_amdgcn_fdot2(a0, b0, acc, false), false);
}

// The lane's query pieces: piece i8 + 8 i of head h (the last one again behind the head).
template <int T, int NP>
__device__ __forceinline__ void load_q(h4 (&qv)[T][NP], const half_t *q, int64_t ldq, int h, int Dh, int i8)
{
#pragma unroll
    for (int i = 0; i < NP; i++)
#pragma unroll
        for (int t = 0; t < T; t++) qv[t][i] = *reinterpret_cast<const h4 *>(q + t * ldq + h * Dh + 4 * min(i8 + 8 * i, Dh / 4 - 1));
}
// ... and zeros there, once the first keys are on their way too
template <int T, int NP>
__device__ __forceinline__ void clear_q(h4 (&qv)[T][NP], int pieces, int i8)
{
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NP; i++)
#pragma unroll
        for (int t = 0; t < T; t++)
            if (i8 + 8 * i >= pieces) qv[t][i] = h4{};
}

// The lane's pieces of the keys j0 + g + NT / 8 it (it < N), of the last one before `end` behind it
template <int NP, int NT, int N>
__device__ __forceinline__ void load_k(h4 (&kv)[N][NP], const half_t *k_head, int64_t ldk, int pieces, int j0, int end)
{
    const int i8 = threadIdx.x & 7, g = threadIdx.x >> 3;
#pragma unroll
    for (int it = 0; it < N; it++)
#pragma unroll
        for (int i = 0; i < NP; i++)
            kv[it][i] = *reinterpret_cast<const h4 *>(k_head + (int64_t)min(j0 + g + it * (NT / 8), end - 1) * ldk +
                                                      4 * min(i8 + 8 * i, pieces - 1));
}
// f16(alpha q . K[j]) for those positions, by the first of a position's lanes to out[t * ldo + j]
template <int T, int NP, int NT, int N>
__device__ __forceinline__ void scores_step(const h4 (&qv)[T][NP], const h4 (&kv)[N][NP], float alpha, int j0, int end, half_t *out,
                                            int64_t ldo)
{
    const int i8 = threadIdx.x & 7, g = threadIdx.x >> 3;
#pragma unroll
    for (int it = 0; it < N; it++)
#pragma unroll
        for (int t = 0; t < T; t++) {
            float a = 0.f;
#pragma unroll
            for (int i = 0; i < NP; i++) a = dot4(qv[t][i], kv[it][i], a);
            a += dpp_f32<0xB1>(a);              // lane ^ 1
            a += dpp_f32<0x4E>(a);              // lane ^ 2
            a += dpp_f32<0x141>(a);             // the other four of the eight
            const int j = j0 + g + it * (NT / 8);
            if (i8 == 0 && j < end) out[t * ldo + j] = f2h(alpha * a);
        }
}

// Values of another workgroup of the same launch, on whatever XCD: past the L2s in both directions, like relaxed atomics of that
// scope, so that there is nothing in a cache to write back or to drop (a device-wide fence does both: 40 us).
__device__ __forceinline__ void store_shared(float *p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float load_shared(const float *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Head h of a launch in parts [h][t][part]: Dh sums, the maximum, the sum of exponentials.
__device__ __forceinline__ void join_parts(int T, int Dh, int nsplit, int h, const float *parts, half_t *out, int64_t ldo)
{
    const int pitch = Dh + 2;
    // exp of a part's maximum less the row's (1 for two infinities of one sign, too)
    auto factor = [](float part, float all) __attribute__((always_inline)) { return part == all ? 1.f : exp_nonpos(fmaxf(part - all, -100.0f)); };
    for (int i = threadIdx.x; i < T * Dh; i += kThreads) {
        const int t = i / Dh, d = i - t * Dh;
        const float *row = parts + ((int64_t)h * T + t) * nsplit * pitch;
        // kJoin parts at a time requested together (the last one again behind them, and left out)
        float mx = -INFINITY, o = 0.f, l = 0.f;
        for (int s0 = 0; s0 < nsplit; s0 += kJoin) {
            float pm[kJoin], pl[kJoin], po[kJoin];
#pragma unroll
            for (int k = 0; k < kJoin; k++) {
                const float *part = row + (int64_t)min(s0 + k, nsplit - 1) * pitch;
                pm[k] = load_shared(part + Dh);
                pl[k] = load_shared(part + Dh + 1);
                po[k] = load_shared(part + d);
            }
            float top = mx;
#pragma unroll
            for (int k = 0; k < kJoin; k++) top = fmaxf(top, pm[k]);
            const float before = factor(mx, top);
            l *= before;
            o *= before;
            mx = top;
#pragma unroll
            for (int k = 0; k < kJoin; k++)
                if (s0 + k < nsplit) {
                    const float f = factor(pm[k], mx);
                    l += f * pl[k];
                    o += f * po[k];
                }
        }
        out[t * ldo + h * Dh + d] = f2h(o / l);
    }
}

// Many positions: a workgroup takes P of them of one head, with all their key and value pieces requested at once, and leaves
// their maximum, the sum of the exponentials against it and that of their products with V; the workgroup of the head that is the
// last to have done so (`arrived`, counters that are 0 when the launch begins) puts them together.  No workgroup waits for
// another.  Without counters the parts are left to decode_join_kernel.  The exponentials stay f32 here, where a row's sum is not
// known before the product with V.
template <int T, int NP, int P>
__global__ void __launch_bounds__(kThreads)
decode_split_kernel(int C, int Dh, int64_t row0, float alpha, const half_t *__restrict__ q, int64_t ldq, const half_t *__restrict__ kc,
                    const half_t *__restrict__ vc, int64_t ldkv, int64_t hs, unsigned *arrived, float *parts, half_t *__restrict__ out, int64_t ldo)
{
    asm volatile("" ::"s"(C), "s"(Dh), "s"(row0), "s"(alpha), "s"(q), "s"(ldq), "s"(kc), "s"(vc), "s"(ldkv), "s"(hs), "s"(arrived), "s"(parts),
                 "s"(out), "s"(ldo));
    constexpr int W = kThreads / 64, LP = 8 * NP, PW = 64 / LP, NV = P / (W * PW);   // lanes per position of V, positions per wave, V pieces of a lane
    static_assert(P % 64 == 0 && NV * W * PW == P, "whole steps");
    __shared__ half_t sp[T][P];
    __shared__ float se[W][T][P];
    __shared__ float red[W][T][4 * LP];
    __shared__ bool last;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, h = blockIdx.x, j0 = blockIdx.y * P, end = min(C, j0 + P), pieces = Dh / 4;
    const int nsplit = gridDim.y;
    const int ip = lane & (LP - 1), g = wid * PW + lane / LP;              // the lane's piece of V, its first position
    const half_t *vp = vc + h * hs + 4 * min(ip, pieces - 1);
    constexpr int KS = P * 8 / kThreads;                                   // positions of a lane in the scores
    h4 qv[T][NP], kv[KS][NP], vv[NV];
    load_q<T, NP>(qv, q, ldq, h, Dh, tid & 7);
    load_k<NP, kThreads>(kv, kc + h * hs, ldkv, pieces, j0, end);
#pragma unroll
    for (int it = 0; it < NV; it++) vv[it] = *reinterpret_cast<const h4 *>(vp + (int64_t)min(j0 + g + it * W * PW, end - 1) * ldkv);
    clear_q<T, NP>(qv, pieces, tid & 7);
    scores_step<T, NP, kThreads>(qv, kv, alpha, 0, end - j0, &sp[0][0], P);
    __syncthreads();
    // every wave works out all statistics: no second barrier, and exponentials of its own in LDS
    float m[T], sum[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
        const int live = (int)min((int64_t)end, (int64_t)t + row0 + 1) - j0;   // of this workgroup's positions
        float s[P / 64];
        m[t] = -INFINITY;
#pragma unroll
        for (int k = 0; k < P / 64; k++) {
            s[k] = h2f(sp[t][lane + 64 * k]);
            if (lane + 64 * k < live) m[t] = fmaxf(m[t], s[k]);
        }
        m[t] = wave_max(m[t]);
        sum[t] = 0.f;
#pragma unroll
        for (int k = 0; k < P / 64; k++) {
            const float e = lane + 64 * k < live ? exp_nonpos(fmaxf(s[k] - m[t], -100.0f)) : 0.f;
            sum[t] += e;
            se[wid][t][lane + 64 * k] = e;
        }
        sum[t] = wave_sum(sum[t]);
    }
    float acc[T][4];
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[t][i] = 0.f;
#pragma unroll
    for (int it = 0; it < NV; it++)
#pragma unroll
        for (int t = 0; t < T; t++) {
            const float e = se[wid][t][g + it * W * PW];
#pragma unroll
            for (int i = 0; i < 4; i++) acc[t][i] += e * h2f(vv[it].v[i]);
        }
#pragma unroll
    for (int t = 0; t < T; t++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (LP <= 16) acc[t][i] = with16(acc[t][i], OpSum());
            acc[t][i] = with32(acc[t][i], OpSum());
        }
        if (lane < LP) *reinterpret_cast<float4_t *>(&red[wid][t][4 * lane]) = float4_t{acc[t][0], acc[t][1], acc[t][2], acc[t][3]};
    }
    __syncthreads();
    // part [h][t][split]: Dh sums, the maximum, the sum of exponentials
    const int pitch = Dh + 2;
    float *mine = parts + ((int64_t)h * T * nsplit + blockIdx.y) * pitch;
    for (int i = tid; i < T * Dh; i += kThreads) {
        const int t = i / Dh, d = i - t * Dh;
        float a = red[0][t][d];
#pragma unroll
        for (int w = 1; w < W; w++) a += red[w][t][d];
        store_shared(mine + (int64_t)t * nsplit * pitch + d, a);
    }
#pragma unroll
    for (int t = 0; t < T; t++)
        if (tid == t) {
            store_shared(mine + (int64_t)t * nsplit * pitch + Dh, m[t]);
            store_shared(mine + (int64_t)t * nsplit * pitch + Dh + 1, sum[t]);
        }
    // every wave's stores have been acknowledged where the other XCDs look, then the count
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (!arrived) return;
    __syncthreads();
    if (tid == 0) last = __hip_atomic_fetch_add(arrived + h * kWordPitch, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)nsplit - 1;
    __syncthreads();
    if (!last) return;
    join_parts(T, Dh, nsplit, h, parts, out, ldo);
}

// The join by itself, behind a split launch without counters.
__global__ void __launch_bounds__(kThreads)
decode_join_kernel(int T, int Dh, int nsplit, const float *parts, half_t *out, int64_t ldo)
{
    join_parts(T, Dh, nsplit, blockIdx.x, parts, out, ldo);
}

// Few positions: a workgroup takes all of them.  LP: lanes per position in the product with V.
template <int T, int NP, int NT, int LP>
__global__ void __launch_bounds__(NT)
decode_values_kernel(int C, int Dh, int64_t row0, float alpha, const half_t *__restrict__ q, int64_t ldq, const half_t *__restrict__ kc,
                     const half_t *__restrict__ vc, int64_t ldkv, int64_t hs, int64_t ld, half_t *__restrict__ out, int64_t ldo)
{
    // the arguments in scalar registers at once (one by one, where first wanted, they are three round trips to memory)
    asm volatile("" ::"s"(C), "s"(Dh), "s"(row0), "s"(alpha), "s"(q), "s"(ldq), "s"(kc), "s"(vc), "s"(ldkv), "s"(hs), "s"(ld),
                 "s"(out), "s"(ldo));
    extern __shared__ __attribute__((aligned(16))) half_t sp[];           // [T][ld]: scores, then probabilities
    __shared__ float scratch[2][T][NT / 64];
    __shared__ float red[NT / 64][T][LP][4];
    constexpr int kGroups = NT / LP;           // positions per step and lane
    const int tid = threadIdx.x, ip = tid & (LP - 1), g = tid / LP, lane = tid & 63, wid = tid >> 6, h = blockIdx.x;
    const int pieces = Dh / 4, per = (pieces + gridDim.y - 1) / gridDim.y;        // pieces of this workgroup: at most LP
    const int piece = blockIdx.y * per + ip;
    const bool mine = ip < per && piece < pieces;
    const half_t *vp = vc + h * hs + 4 * (mine ? piece : 0);
    auto load_v = [&](h4 (&v)[kStep], int j0) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < kStep; it++)
            v[it] = *reinterpret_cast<const h4 *>(vp + (int64_t)min(j0 + g + it * kGroups, C - 1) * ldkv);
    };
    h4 vv[kStep];
    h4 qv[T][NP], kv[kStep][NP];
    load_q<T, NP>(qv, q, ldq, h, Dh, tid & 7);
    load_k<NP, NT>(kv, kc + h * hs, ldkv, pieces, 0, C);
    load_v(vv, 0);
    clear_q<T, NP>(qv, pieces, tid & 7);
    scores_step<T, NP, NT>(qv, kv, alpha, 0, C, sp, ld);
    for (int j0 = NT / 8 * kStep; j0 < C; j0 += NT / 8 * kStep) {
        load_k<NP, NT>(kv, kc + h * hs, ldkv, pieces, j0, C);
        scores_step<T, NP, NT>(qv, kv, alpha, j0, C, sp, ld);
    }
    __syncthreads();
    // position tid + k NT of row t, k < KMAX: its score, then its exponential, held by the lane
    constexpr int KMAX = NT == kThreads ? 1 : 2;
    static_assert((NT == kThreads ? kNarrow : kOwnScoresShort) <= KMAX * NT, "a row's scores in registers");
    float e[T][KMAX], m[T], sum[T];
    auto live = [&](int t) __attribute__((always_inline)) { return (int)min((int64_t)C, (int64_t)t + row0 + 1); };
    // row maxima, then sums of exponentials, then the probabilities; row t sees live(t) positions
#pragma unroll
    for (int t = 0; t < T; t++) {
        m[t] = -INFINITY;
#pragma unroll
        for (int k = 0; k < KMAX; k++) {
            const int j = tid + k * NT;
            e[t][k] = h2f(sp[t * ld + min(j, C - 1)]);
            if (j < live(t)) m[t] = fmaxf(m[t], e[t][k]);
        }
        m[t] = wave_max(m[t]);
        if (lane == 0) scratch[0][t][wid] = m[t];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < T; t++) {
        m[t] = scratch[0][t][0];
#pragma unroll
        for (int w = 1; w < NT / 64; w++) m[t] = fmaxf(m[t], scratch[0][t][w]);
        sum[t] = 0.f;
#pragma unroll
        for (int k = 0; k < KMAX; k++) {
            e[t][k] = exp_nonpos(fmaxf(e[t][k] - m[t], -100.0f));
            if (tid + k * NT < live(t)) sum[t] += e[t][k];
        }
        sum[t] = wave_sum(sum[t]);
        if (lane == 0) scratch[1][t][wid] = sum[t];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < T; t++) {
        sum[t] = scratch[1][t][0];
#pragma unroll
        for (int w = 1; w < NT / 64; w++) sum[t] += scratch[1][t][w];
        const RowDivide div(sum[t]);
#pragma unroll
        for (int k = 0; k < KMAX; k++) {
            const int j = tid + k * NT;
            if (j < C) sp[t * ld + j] = j < live(t) ? f2h(div(e[t][k])) : (half_t)0.f;
        }
    }
    __syncthreads();
    float acc[T][4];
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[t][i] = 0.f;
    auto add = [&](int j0) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < kStep; it++) {
            const int j = j0 + g + it * kGroups;
#pragma unroll
            for (int t = 0; t < T; t++) {
                const float p = j < C ? h2f(sp[t * ld + j]) : 0.f;
#pragma unroll
                for (int i = 0; i < 4; i++) acc[t][i] += p * h2f(vv[it].v[i]);
            }
        }
    };
    int j0 = 0;
    for (; j0 + kGroups * kStep < C; j0 += kGroups * kStep) {
        h4 vn[kStep];
        load_v(vn, j0 + kGroups * kStep);
        add(j0);
#pragma unroll
        for (int it = 0; it < kStep; it++) vv[it] = vn[it];
    }
    add(j0);                                  // (without a request behind it, which would be waited for)
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float a = acc[t][i];
            if (LP <= 2) a += dpp<0x4E>(a);                 // lane ^ 2
            if (LP <= 4) a += dpp<0x1B>(dpp<0x141>(a));     // lane ^ 7 ^ 3
            a += dpp<0x128>(a);                             // row_ror 8: lane ^ 8
            a = with32(with16(a, OpSum()), OpSum());
            if (lane < LP) red[wid][t][lane][i] = a;
        }
    __syncthreads();
    if (tid < T * LP * 4) {
        const int t = tid / (LP * 4), c = (tid >> 2) & (LP - 1), i = tid & 3;
        if (c < per && blockIdx.y * per + c < pieces) {
            float a = red[0][t][c][i];
#pragma unroll
            for (int w = 1; w < NT / 64; w++) a += red[w][t][c][i];
            out[t * ldo + h * Dh + 4 * (blockIdx.y * per + c) + i] = f2h(a);
        }
    }
}

struct DecodeArgs {
    int C, H, Dh;
    int64_t row0;
    float alpha;
    const half_t *q;
    int64_t ldq;
    const half_t *kc, *vc;
    int64_t ldkv, hs;
    half_t *out;
    int64_t ldo;
    void *ws;
    bool cleared;
    hipStream_t st;
};

template <int T, int NP, int NT, int LP>
int launch_values(const DecodeArgs &a)
{
    const int64_t ld = (a.C + 7) / 8 * 8;
    hipLaunchKernelGGL((decode_values_kernel<T, NP, NT, LP>), dim3((unsigned)a.H, (unsigned)((a.Dh / 4 + LP - 1) / LP)), dim3(NT),
                       (size_t)T * (size_t)ld * sizeof(half_t), a.st, a.C, a.Dh, a.row0, a.alpha, a.q, a.ldq, a.kc, a.vc, a.ldkv, a.hs, ld, a.out, a.ldo);
    return launch_status("attn_decode");
}

// positions of a row up to which a workgroup takes them all
int64_t most_in_one(int64_t T, int64_t Dh, bool cleared)
{
    return Dh > 64 ? (cleared ? kOwnScoresCleared : kOwnScores) : T > 2 ? kOwnScores : cleared ? kOwnScoresShortCleared : kOwnScoresShort;
}
int64_t split_words(int64_t H) { return H * kWordPitch; }

template <int T, int NP, int P>
int launch_split(const DecodeArgs &a)
{
    const int nsplit = (a.C + P - 1) / P;
    unsigned *words = static_cast<unsigned *>(a.ws);
    float *parts = reinterpret_cast<float *>(words) + split_words(a.H);
    hipLaunchKernelGGL((decode_split_kernel<T, NP, P>), dim3((unsigned)a.H, (unsigned)nsplit), dim3(kThreads), 0, a.st, a.C, a.Dh, a.row0,
                       a.alpha, a.q, a.ldq, a.kc, a.vc, a.ldkv, a.hs, a.cleared ? words : nullptr, parts, a.out, a.ldo);
    if (!a.cleared) hipLaunchKernelGGL(decode_join_kernel, dim3((unsigned)a.H), dim3(kThreads), 0, a.st, T, a.Dh, nsplit, parts, a.out, a.ldo);
    return launch_status("attn_decode");
}

template <int T, int NP>
int launch(const DecodeArgs &a)
{
    if (a.C <= kNarrow) return launch_values<T, NP, kThreads, 8>(a);
    if (a.C <= most_in_one(T, a.Dh, a.cleared)) return launch_values<T, NP, kWide, 4>(a);
    if (a.C <= kJoin * 64) return launch_split<T, NP, 64>(a);
    if (a.C <= kJoin * 128) return launch_split<T, NP, 128>(a);
    return launch_split<T, NP, 256>(a);
}

template <int NP>
int launch_rows(int64_t T, const DecodeArgs &a)
{
    return T == 1 ? launch<1, NP>(a) : T == 2 ? launch<2, NP>(a) : T == 3 ? launch<3, NP>(a) : launch<4, NP>(a);
}

}  // namespace

namespace cacti {

// Words, kClearPitch apart, from the start of the workspace on that a launch over C positions wants to be 0: one that has `cleared`
// them, in front of it on the stream, saves the launch that does it.
int64_t attn_decode_words(int64_t T, int64_t H, int64_t Dh, int64_t C) { return C <= most_in_one(T, Dh, true) ? 0 : H; }

int attn_decode(int64_t T, int64_t H, int64_t Dh, int64_t C, int64_t initial_row, float alpha, const void *q, int64_t ldq, const void *k_cache,
                const void *v_cache, int64_t ldkv, int64_t head_stride, void *out, int64_t ldo, void *workspace, size_t workspace_bytes, bool cleared,
                hipStream_t st)
{
    CACTI_REQUIRE(T >= 1 && T <= 4 && H > 0 && H <= 65535 && C > 0 && initial_row >= 0, CACTI_E_NOTIMPL,
                  "attn_decode: 1 to 4 rows are handled here (T=%lld)", (long long)T);
    CACTI_REQUIRE(Dh % 4 == 0 && Dh >= 4 && Dh <= 128, CACTI_E_NOTIMPL, "attn_decode: need Dh %% 4 == 0 and Dh <= 128");
    CACTI_REQUIRE(q && k_cache && v_cache && out && workspace, CACTI_E_INVALID, "attn_decode: null pointer");
    CACTI_REQUIRE(C <= kMaxCols, CACTI_E_NOTIMPL, "attn_decode: at most %d cached positions", kMaxCols);
    CACTI_REQUIRE(ldq % 4 == 0 && ldkv % 4 == 0 && head_stride % 4 == 0 && aligned(q, 8) && aligned(k_cache, 8) && aligned(v_cache, 8) &&
                      aligned(workspace, 16),
                  CACTI_E_INVALID, "attn_decode: operands must be 8-byte aligned with row pitches that are multiples of 4");
    CACTI_REQUIRE(workspace_bytes >= cacti_hip_attn_decode_workspace(T, H, Dh, C), CACTI_E_INVALID,
                  "attn_decode: workspace too small");
    // columns beyond the last row's position are masked for every row: they are not formed
    const int64_t live = C < T + initial_row ? C : T + initial_row;
    const DecodeArgs a = {(int)live, (int)H, (int)Dh, initial_row, alpha, (const half_t *)q, ldq, (const half_t *)k_cache,
                          (const half_t *)v_cache, ldkv, head_stride, (half_t *)out, ldo, workspace, cleared, st};
    return Dh <= 64 ? launch_rows<2>(T, a) : launch_rows<4>(T, a);
}

}  // namespace cacti

CACTI_API size_t cacti_hip_attn_decode_workspace(int64_t T, int64_t H, int64_t Dh, int64_t C)
{
    if (T <= 0 || H <= 0 || Dh <= 0 || C <= 0) return 0;
    // as many parts as C positions or fewer have (of 64, 128 or 256)
    const int64_t parts = std::max(std::min<int64_t>(kJoin, (C + 63) / 64), (C + 255) / 256);
    return sizeof(float) * (size_t)(split_words(H) + T * H * parts * (Dh + 2));
}

CACTI_API int cacti_hip_attn_decode_f16(int64_t T, int64_t H, int64_t Dh, int64_t C, int64_t initial_row, float alpha,
                                        const void *q, int64_t ldq, const void *k_cache, const void *v_cache,
                                        int64_t ldkv, int64_t head_stride, void *out, int64_t ldo, void *workspace,
                                        size_t workspace_bytes, void *stream)
{
    return attn_decode(T, H, Dh, C, initial_row, alpha, q, ldq, k_cache, v_cache, ldkv, head_stride, out, ldo, workspace, workspace_bytes, false,
                       (hipStream_t)stream);
}
