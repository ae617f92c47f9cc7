// Attention of one to four new positions over the key / value cache (decoding): the chain
//   block_matmul_scale(q, k_cache^T, 1/sqrt(Dh)) -> f32 -> row-causal mask -> softmax -> f16
//   -> block_matmul(., v_cache)                      src/librarium/llama.rs:895-915
// with the reference's rounding points (scores and probabilities are f16 values, both products
// accumulate in fp32 and round once).
//
// A single query row per head is a few hundred KB of cache and hardly any arithmetic: what it costs is launches and
// round trips to memory.  A workgroup takes a head and a piece of its dimension (8 to 32 columns), over all positions:
// the probabilities of a row need the sum over the whole row before the first product with V is formed, and a split
// over positions would need that sum, and then the partial outputs, exchanged between workgroups (another launch each;
// a device-wide fence inside the launch costs 40 us on this chip).  Every piece's workgroup forms the head's scores
// itself, K coming out of L2 for all but the first; from kOwnScores positions on, where that would be most of the
// time, the scores come from a launch of their own, one workgroup per head and 128 positions.  One launch instead of
// three (scores, values per 128 positions, sum): 69 positions, 32 heads of 100: 12.9 -> 5 us.
//
// In the scores eight lanes share a position, each with 8-byte pieces of the head (a head starts on a multiple of 8
// bytes), 64 contiguous bytes per access; in the product with V it is LP lanes with a piece each: fewer columns per
// workgroup are more workgroups, each with fewer steps over the positions behind one another.  (The head is the fast
// index of the grid: where their number is a multiple of 8, all workgroups of a head are on one XCD and share a row's
// bytes in its L2.)  Four positions per lane are in flight together; the first V pieces are requested once the scores'
// own loads are, which would otherwise be returned behind them, and arrive during the softmax.  Loads are unconditional
// with clamped indices: a load inside a branch is waited for at the end of the branch.
// Eight lanes throughout and V first -> now, us: one row, 16 heads of 128, 200 / 480 / 1540 / 4000 positions 5.7 / 6.8 /
// 10.7 / 18.5 -> 5.0 / 6.1 / 8.9 / 15.4; 32 heads of 100 6.5 / 9.3 / 16.2 / 31.6 -> 5.6 / 7.2 / 12.5 / 23.0; four rows of
// 16 x 128 10.9 / 13.3 / 20.1 / 35.7 -> 10.4 / 12.6 / 16.9 / 26.7 (before the exponentials were held by the lanes).
#include "common.h"
#include "softmax_math.h"

using namespace cacti;

namespace {

constexpr int kThreads = 256;              // of the scores launch; the values launch has kThreads or kWide
constexpr int kWide = 512;
constexpr int kStep = 4;                   // positions of a lane in flight
constexpr int kSlice = kThreads / 8 * kStep;   // positions per workgroup of the scores launch
// Up to here kThreads lanes, eight to a position, own scores: one step over the positions, which more lanes cannot make
// shorter (70 positions, 32 heads of 100: 4.6 against 4.9 us; 300 positions 6.8 against 6.5).
constexpr int kNarrow = 128;
// Up to here kWide lanes, four to a position, own scores; beyond, a scores launch: 16 heads of 128, 400 / 520 / 800
// positions 6.1 / 7.5 / 8.6 against 6.8 / 7.0 / 7.3 us, 32 heads of 100 6.8 / 8.2 / 9.7 against 6.9 / 7.8 / 8.6.
constexpr int kOwnScores = 480;
// The same for one or two rows of heads to 64, which have half of the keys' bytes to read: 32 heads of 64, 800 / 1200
// positions 6.9 / 8.3 against 7.7 / 8.1 us; four rows of 16 such heads at 520 13.0 against 12.9.
constexpr int kOwnScoresShort = 960;
constexpr int kMaxCols = 8192;             // score rows live in LDS

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

// The lane's pieces of the keys j0 + g + NT / 8 it (it < kStep), of the last one before `end` behind it
template <int NP, int NT>
__device__ __forceinline__ void load_k(h4 (&kv)[kStep][NP], const half_t *k_head, int64_t ldk, int pieces, int j0, int end)
{
    const int i8 = threadIdx.x & 7, g = threadIdx.x >> 3;
#pragma unroll
    for (int it = 0; it < kStep; it++)
#pragma unroll
        for (int i = 0; i < NP; i++)
            kv[it][i] = *reinterpret_cast<const h4 *>(k_head + (int64_t)min(j0 + g + it * (NT / 8), end - 1) * ldk +
                                                      4 * min(i8 + 8 * i, pieces - 1));
}
// f16(alpha q . K[j]) for those positions, by the first of a position's lanes to out[t * ldo + j]
template <int T, int NP, int NT>
__device__ __forceinline__ void scores_step(const h4 (&qv)[T][NP], const h4 (&kv)[kStep][NP], float alpha, int j0, int end, half_t *out,
                                            int64_t ldo)
{
    const int i8 = threadIdx.x & 7, g = threadIdx.x >> 3;
#pragma unroll
    for (int it = 0; it < kStep; it++)
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

template <int T, int NP>
__global__ void __launch_bounds__(kThreads)
decode_scores_kernel(int C, int Dh, float alpha, const half_t *__restrict__ q, int64_t ldq, const half_t *__restrict__ kc, int64_t ldk,
                     int64_t hsk, half_t *__restrict__ s16, int64_t ld)
{
    asm volatile("" ::"s"(C), "s"(Dh), "s"(alpha), "s"(q), "s"(ldq), "s"(kc), "s"(ldk), "s"(hsk), "s"(s16), "s"(ld));
    const int h = blockIdx.y, j0 = blockIdx.x * kSlice, end = min(C, j0 + kSlice);
    h4 qv[T][NP], kv[kStep][NP];
    load_q<T, NP>(qv, q, ldq, h, Dh, threadIdx.x & 7);
    load_k<NP, kThreads>(kv, kc + h * hsk, ldk, Dh / 4, j0, end);
    clear_q<T, NP>(qv, Dh / 4, threadIdx.x & 7);
    scores_step<T, NP, kThreads>(qv, kv, alpha, j0, end, s16 + (int64_t)h * T * ld, ld);
}

// OWN: the scores are formed here; otherwise they are s16[h][t][ld].  LP: lanes per position in the product with V.
template <int T, int NP, bool OWN, int NT, int LP>
__global__ void __launch_bounds__(NT)
decode_values_kernel(int C, int Dh, int64_t row0, float alpha, const half_t *__restrict__ q, int64_t ldq, const half_t *__restrict__ kc,
                     const half_t *__restrict__ vc, int64_t ldkv, int64_t hs, const half_t *__restrict__ s16, int64_t ld,
                     half_t *__restrict__ out, int64_t ldo)
{
    // the arguments in scalar registers at once (one by one, where first wanted, they are three round trips to memory)
    asm volatile("" ::"s"(C), "s"(Dh), "s"(row0), "s"(alpha), "s"(q), "s"(ldq), "s"(kc), "s"(vc), "s"(ldkv), "s"(hs), "s"(s16), "s"(ld),
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
    if (OWN) {
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
    } else {
        for (int i = tid; i < T * (int)ld / 8; i += NT) st8(sp + i * 8, ld8(s16 + (int64_t)h * T * ld + i * 8));
        load_v(vv, 0);
    }
    __syncthreads();
    // position tid + k NT of row t, k < KMAX: its score, then its exponential, held by the lane.  They cover a whole row of own
    // scores and one of 2048 positions; behind them the scores are read again and the exponentials formed twice, as they were
    // everywhere: 1540 positions of 16 heads of 128 6.2 -> 5.0 us, 2000 of 32 of 100 9.1 -> 7.8, 70 4.5 -> 4.2, four rows of 16 of
    // 128 over 200 11.0 -> 9.0.  (All that a row can have held is code that a launch fetches in vain: 700 positions of 32 heads
    // of 100 5.0 -> 5.8 us; with four 4.4.)
    constexpr int KMAX = !OWN ? 4 : NT == kThreads ? 1 : 2;
    static_assert(!OWN || (NT == kThreads ? kNarrow : kOwnScoresShort) <= KMAX * NT, "a row's own scores in registers");
    float e[T][KMAX], m[T], sum[T];
    auto live = [&](int t) __attribute__((always_inline)) { return (int)min((int64_t)C, (int64_t)t + row0 + 1); };
    auto more = [&](int t, int end, auto &&f) __attribute__((always_inline)) {
        if constexpr (!OWN)
            for (int j = tid + KMAX * NT; j < end; j += NT) f(sp + t * ld + j, j);
    };
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
        more(t, live(t), [&](half_t *s, int) __attribute__((always_inline)) { m[t] = fmaxf(m[t], h2f(*s)); });
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
        more(t, live(t), [&](half_t *s, int) __attribute__((always_inline)) { sum[t] += exp_nonpos(fmaxf(h2f(*s) - m[t], -100.0f)); });
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
        more(t, C, [&](half_t *s, int j) __attribute__((always_inline)) {
            *s = j < live(t) ? f2h(div(exp_nonpos(fmaxf(h2f(*s) - m[t], -100.0f)))) : (half_t)0.f;
        });
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
    half_t *s16;
    hipStream_t st;
};

template <int T, int NP, bool OWN, int NT, int LP>
int launch_values(const DecodeArgs &a, int64_t ld)
{
    const size_t smem = (size_t)T * (size_t)ld * sizeof(half_t);
    auto kern = decode_values_kernel<T, NP, OWN, NT, LP>;
    if (smem > 32 * 1024) {
        static DeviceOnce attr_set;
        if (!attr_set.fresh()) {
            CACTI_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, T * kMaxCols * (int)sizeof(half_t)));
            attr_set.mark();
        }
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)a.H, (unsigned)((a.Dh / 4 + LP - 1) / LP)), dim3(NT), smem, a.st, a.C, a.Dh, a.row0, a.alpha, a.q,
                       a.ldq, a.kc, a.vc, a.ldkv, a.hs, (const half_t *)a.s16, ld, a.out, a.ldo);
    return launch_status("attn_decode");
}

template <int T, int NP>
int launch(const DecodeArgs &a)
{
    const int64_t ld = (a.C + 7) / 8 * 8;
    if (a.C <= kNarrow) return launch_values<T, NP, true, kThreads, 8>(a, ld);
    if (a.C <= (NP == 2 && T <= 2 ? kOwnScoresShort : kOwnScores)) return launch_values<T, NP, true, kWide, 4>(a, ld);
    hipLaunchKernelGGL((decode_scores_kernel<T, NP>), dim3((unsigned)((a.C + kSlice - 1) / kSlice), (unsigned)a.H), dim3(kThreads), 0, a.st,
                       a.C, a.Dh, a.alpha, a.q, a.ldq, a.kc, a.ldkv, a.hs, a.s16, ld);
    // two lanes to a position while every workgroup of theirs has a CU (1540 positions, 16 heads of 128, two / four: 8.8 /
    // 9.3 us, 32 of 64 8.9 / 9.6; 32 of 100, 416 workgroups, 14.0 / 12.2)
    if ((int64_t)a.H * ((a.Dh / 4 + 1) / 2) <= device_cus()) return launch_values<T, NP, false, kWide, 2>(a, ld);
    return launch_values<T, NP, false, kWide, 4>(a, ld);
}

template <int NP>
int launch_rows(int64_t T, const DecodeArgs &a)
{
    return T == 1 ? launch<1, NP>(a) : T == 2 ? launch<2, NP>(a) : T == 3 ? launch<3, NP>(a) : launch<4, NP>(a);
}

}  // namespace

CACTI_API size_t cacti_hip_attn_decode_workspace(int64_t T, int64_t H, int64_t Dh, int64_t C)
{
    if (T <= 0 || H <= 0 || Dh <= 0 || C <= 0) return 0;
    return (size_t)(T * H * ((C + 7) / 8 * 8) * 2);               // scores [H, T, C rounded up] f16
}

CACTI_API int cacti_hip_attn_decode_f16(int64_t T, int64_t H, int64_t Dh, int64_t C, int64_t initial_row, float alpha,
                                        const void *q, int64_t ldq, const void *k_cache, const void *v_cache,
                                        int64_t ldkv, int64_t head_stride, void *out, int64_t ldo, void *workspace,
                                        size_t workspace_bytes, void *stream)
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
                          (const half_t *)v_cache, ldkv, head_stride, (half_t *)out, ldo, (half_t *)workspace, (hipStream_t)stream};
    return Dh <= 64 ? launch_rows<2>(T, a) : launch_rows<4>(T, a);
}
