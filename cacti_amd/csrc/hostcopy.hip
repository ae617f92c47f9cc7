// Data on its way from the device to the host program, and many small regions cleared at once.
//
// A read-back of a few KB costs its round trips, not its bytes: hipMemcpyAsync into pageable memory is staged by the
// runtime and a stream synchronisation takes some 15 us to notice that the stream is empty.  Here one kernel writes the
// regions straight into page-locked host memory in chunks, each followed by a word that says it is there, and the host
// polls those words.  Of a large read the host copies the chunks that have arrived to their place while the others are on
// the link (the runtime's copy to pageable memory: 16 GB/s).
#include <emmintrin.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <mutex>

#include "chunks.h"
#include "common.h"
#include "hostcopy.h"

namespace cacti {

namespace {

constexpr int kGatherBlocks = 64;              // chunks per region of a small read at most: 4 KB and more each
constexpr int kFlagsPerGather = kGatherBlocks * kMaxRegions;
static_assert(kFlagsPerGather * sizeof(unsigned) <= Staging::kFlagBytes, "a word per workgroup");

struct GatherArgs {
    const uint4 *src[kMaxRegions];
    uint4 *dst[kMaxRegions];
    int64_t n16[kMaxRegions];
    unsigned *flags;
    unsigned epoch;
};

// Sixteen bytes to host memory at system scope: through both caches, like a relaxed atomic of that scope (which the language
// has for eight bytes at most).  So there is nothing in the caches for a system fence to write back before the word that
// announces the chunk, only stores to wait for; the fence, once per wave, was a third of the read (64 KiB 12.0 -> 9.0 us,
// 344 KiB 24.7 -> 18.2 from launch to copied, 64 bytes 6.9 -> 5.8).
__device__ __forceinline__ void store_host(uint4 *dst, const uint4 &v)
{
    typedef unsigned uint4_v __attribute__((ext_vector_type(4)));
    const uint4_v w = {v.x, v.y, v.z, v.w};
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" : : "v"(dst), "v"(w) : "memory");
}
__device__ __forceinline__ void store_host(int *dst, int v)
{
    __hip_atomic_store(dst, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// every wave's stores have been acknowledged, then the word
__device__ __forceinline__ void chunk_arrived(unsigned *flag, unsigned epoch)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(flag, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void __launch_bounds__(256) gather_kernel(GatherArgs p)
{
    const int z = blockIdx.y;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < p.n16[z]; i += (int64_t)gridDim.x * 256) store_host(p.dst[z] + i, p.src[z][i]);
    chunk_arrived(p.flags + z * gridDim.x + blockIdx.x, p.epoch);
}

// One large region.  The link is full with a few workgroups (16: 52 GB/s); more of them would only make the chunks
// arrive all together at the end, and the host wants them one after another.
__global__ void __launch_bounds__(256)
stream_kernel(const uint4 *src, uint4 *dst, int64_t n16, int64_t chunk16, const int *word, int *word_dst, unsigned *flags, unsigned epoch)
{
    const int64_t chunks = (n16 + chunk16 - 1) / chunk16;
    for (int64_t c = blockIdx.x; c < chunks; c += gridDim.x) {
        if (word && c == 0 && threadIdx.x == 0) store_host(word_dst, *word);
        const int64_t end = min((c + 1) * chunk16, n16);
        for (int64_t i = c * chunk16 + threadIdx.x; i < end; i += 256) store_host(dst + i, src[i]);
        chunk_arrived(flags + c, epoch);
    }
}

struct ZeroArgs {
    uint4 *p[kMaxRegions];
    int64_t n16;
};

__global__ void __launch_bounds__(256) zero_regions_kernel(ZeroArgs a)
{
    uint4 *p = a.p[blockIdx.y];
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.n16; i += (int64_t)gridDim.x * 256) p[i] = make_uint4(0, 0, 0, 0);
}

int launch_gather(const HostRegion *r, int n, unsigned *flags, unsigned epoch, int *nflags, hipStream_t st)
{
    GatherArgs p = {};
    int64_t most = 1;
    for (int i = 0; i < n; i++) {
        p.src[i] = static_cast<const uint4 *>(r[i].src);
        p.dst[i] = static_cast<uint4 *>(r[i].dst);
        p.n16[i] = (int64_t)((r[i].bytes + 15) / 16);
        most = std::max(most, p.n16[i]);
    }
    p.flags = flags;
    p.epoch = epoch;
    const int blocks = (int)std::min<int64_t>((most + 255) / 256, kGatherBlocks);
    *nflags = blocks * n;
    hipLaunchKernelGGL(gather_kernel, dim3((unsigned)blocks, (unsigned)n), dim3(256), 0, st, p);
    return launch_status("gather_to_host");
}

// until all words hold `epoch`; a stream that is busy for longer than polling is worth is waited for by the runtime,
// which also reports a failed one
int wait_flags(const unsigned *flags, int n, unsigned epoch, hipStream_t st)
{
    const auto begin = std::chrono::steady_clock::now();
    int i = 0;
    for (unsigned polls = 1;; polls++) {
        while (i < n && __atomic_load_n(flags + i, __ATOMIC_ACQUIRE) == epoch) i++;
        if (i == n) return 0;
        _mm_pause();
        if ((polls & 255) == 0 && std::chrono::steady_clock::now() - begin > std::chrono::milliseconds(50)) break;
    }
    CACTI_HIP(hipStreamSynchronize(st));
    for (; i < n; i++)
        CACTI_REQUIRE(__atomic_load_n(flags + i, __ATOMIC_ACQUIRE) == epoch, CACTI_E_STATE, "gather_to_host: a part did not arrive");
    return 0;
}

// Buffers nobody uses at the moment, by size: at most 4 of a context's, for the next contexts, 16 of a word's, one for
// every thread that reads at the same time, and two windows of reads above kOwnRead (a third such reader at the same time
// page-locks its own and frees it again).
struct Kept {
    size_t bytes;
    int most, n;
    Staging free[16];
    Staging take(int i)
    {
        const Staging s = free[i];
        free[i] = free[--n];
        return s;
    }
};
std::mutex g_mutex;
Kept g_kept[] = {{kStagingBytes, 4, 0, {}}, {kWordBytes, 16, 0, {}}, {kWindowBytes, 2, 0, {}}};
std::atomic<size_t> g_pinned{0};               // bytes page-locked here, kept or in use
unsigned g_resets[64];                         // per device, under g_mutex

Kept *kept_of(size_t bytes)
{
    for (Kept &k : g_kept)
        if (k.bytes == bytes) return &k;
    return nullptr;
}

void *pinned_alloc(size_t bytes)
{
    void *p = nullptr;
    if (hipHostMalloc(&p, bytes, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    g_pinned += bytes;
    return p;
}
void pinned_free(void *p, size_t bytes)
{
    hipHostFree(p);
    g_pinned -= bytes;
}

// After a failure: the kernel may still be writing the buffer.  Where not even waiting for it works, the buffer is never
// handed out again.
void settle(Staging &s, hipStream_t st)
{
    if (hipStreamSynchronize(st) == hipSuccess) return;
    (void)hipGetLastError();
    s.lost = true;
}

// a large read's buffer: a word per chunk, at the end of their place the word that is read with it (a gather's words, in the
// same buffer, do not reach there), then the window of chunks
constexpr size_t kWindow = kWindowBytes - Staging::kFlagBytes, kLeastChunk = 16u << 10, kWordPlace = Staging::kFlagBytes - 64;
static_assert((1u << 20) / kLeastChunk * sizeof(unsigned) <= kWordPlace && kWindow / (2 * kLeastChunk) * sizeof(unsigned) <= kWordPlace && kFlagsPerGather * sizeof(unsigned) <= kWordPlace,
              "a word per chunk");
constexpr int kStreamBlocks = 16;

}  // namespace

int gather_to_host(Staging &s, const HostRegion *r, int n, hipStream_t st)
{
    CACTI_REQUIRE(n >= 1 && n <= kMaxRegions, CACTI_E_INVALID, "gather_to_host: %d regions", n);
    unsigned *flags = reinterpret_cast<unsigned *>(s.base);
    int nflags = 0;
    if (++s.epoch == 0) s.epoch = 1;
    int rc = launch_gather(r, n, flags, s.epoch, &nflags, st);
    if (rc) return rc;
    rc = wait_flags(flags, nflags, s.epoch, st);
    if (rc) settle(s, st);
    return rc;
}

static int read_windows(Staging &s, void *dst, const void *src, size_t bytes, const int *word, int *word_dst, hipStream_t st)
{
    int *const word_here = reinterpret_cast<int *>(s.base + kWordPlace);
    unsigned *const flags = reinterpret_cast<unsigned *>(s.base);
    char *const data = s.data();
    int dev = 0;
    CACTI_HIP(hipGetDevice(&dev));
    for (size_t done = 0; done < bytes;) {
        const size_t window = std::min(bytes - done, s.room()), chunk = window <= (1u << 20) ? kLeastChunk : window < (4u << 20) ? 2 * kLeastChunk : 4 * kLeastChunk;
        const int chunks = (int)((window + chunk - 1) / chunk), threads = (int)std::min<size_t>(kCopyThreads, 1 + window / (4u << 20));
        if (++s.epoch == 0) s.epoch = 1;
        const unsigned epoch = s.epoch;
        hipLaunchKernelGGL(stream_kernel, dim3((unsigned)std::min(chunks, kStreamBlocks)), dim3(256), 0, st,
                           reinterpret_cast<const uint4 *>(static_cast<const char *>(src) + done), reinterpret_cast<uint4 *>(data),
                           (int64_t)((window + 15) / 16), (int64_t)(chunk / 16), word, word_here, flags, epoch);
        const int rc = launch_status("read_large");
        if (rc) return rc;
        const ChunkError e = copy_chunks(
            static_cast<char *>(dst) + done, data, window, chunk, threads, [&]() { (void)hipSetDevice(dev); },
            [&](int i) { return wait_flags(flags + i, 1, epoch, st); }, []() { return cacti_hip_last_error(); });
        if (e.rc) {
            settle(s, st);
            set_error("%s", e.text);
            return e.rc;
        }
        done += window;
    }
    if (word) *word_dst = *word_here;
    return 0;
}

// Measured, us, one gather and one copy behind it / 1 MiB pieces before -> chunks: 2 MiB 119 -> 76, 20 MiB 569 -> 473.  A
// helper thread costs some 10 us to start: worth it from several MiB on, where the copying host (12 .. 30 GB/s) and not
// the link (52) is what one thread would wait for.  One gather and one copy behind it against chunks, since the chunks are
// announced without a fence: 128 KiB 15.3 and 15.7, 344 KiB 24.4 and 22.3, 512 KiB 30.2 and 29.6.  Up to 1 MiB in chunks of
// 16 KiB, so that the 16 workgroups have some one after another and the host a copy to make meanwhile: 128 KiB (one gather
// before) 14.4 -> 13.6, 512 KiB 29.0 -> 25.7; in chunks of 8 KiB 15.3 and 27.2, by 32 workgroups 13.6 and 30.2.
int read_large(Staging &own, void *dst, const void *src, size_t bytes, const int *word, int *word_dst, hipStream_t st)
{
    if (own.base && !own.lost && bytes <= kOwnRead) return read_windows(own, dst, src, bytes, word, word_dst, st);
    Staging s;
    if (!staging_take(&s, kWindowBytes)) {
        CACTI_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
        if (word) CACTI_HIP(hipMemcpyAsync(word_dst, word, sizeof(int), hipMemcpyDeviceToHost, st));
        CACTI_HIP(hipStreamSynchronize(st));
        return 0;
    }
    const int rc = read_windows(s, dst, src, bytes, word, word_dst, st);
    staging_give_back(&s);
    return rc;
}

int zero_regions(void *const *ptrs, int n, size_t bytes, hipStream_t st)
{
    for (int i0 = 0; i0 < n; i0 += kMaxRegions) {
        ZeroArgs a = {};
        const int m = std::min(n - i0, kMaxRegions);
        for (int i = 0; i < m; i++) a.p[i] = static_cast<uint4 *>(ptrs[i0 + i]);
        a.n16 = (int64_t)(bytes / 16);
        const unsigned blocks = (unsigned)std::min<int64_t>((a.n16 + 255) / 256, 512);
        hipLaunchKernelGGL(zero_regions_kernel, dim3(blocks, (unsigned)m), dim3(256), 0, st, a);
        const int rc = launch_status("zero_regions");
        if (rc) return rc;
    }
    return 0;
}

bool staging_take(Staging *s, size_t bytes)
{
    Kept *k = kept_of(bytes);
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
        (void)hipGetLastError();
        return false;
    }
    *s = Staging{};
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        for (int i = k->n; i-- > 0;)
            if (k->free[i].dev == dev) {
                *s = k->take(i);
                return true;
            }
        s->resets = g_resets[dev];
    }
    void *p = pinned_alloc(bytes);
    if (!p) return false;
    memset(p, 0, Staging::kFlagBytes);
    s->base = static_cast<char *>(p);
    s->bytes = bytes;
    s->dev = dev;
    return true;
}

void staging_give_back(Staging *s)
{
    if (!s->base) return;
    bool keep = false, ours;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        Kept *k = kept_of(s->bytes);
        ours = !s->lost && s->resets == g_resets[s->dev];
        keep = ours && k->n < k->most;
        if (keep) k->free[k->n++] = *s;
    }
    // (one that may still be written, or that a reset has deleted, is neither kept nor freed)
    if (ours && !keep) pinned_free(s->base, s->bytes);
    else if (!ours && !s->lost) g_pinned -= s->bytes;
    *s = Staging{};
}

void staging_release(int dev)
{
    if (dev < 0 || dev >= 64) return;
    std::lock_guard<std::mutex> lock(g_mutex);
    for (Kept &k : g_kept)
        for (int i = k.n; i-- > 0;)
            if (k.free[i].dev == dev) pinned_free(k.take(i).base, k.bytes);
    g_resets[dev]++;
}

}  // namespace cacti

using namespace cacti;

// The buffer is the call's, not the thread's: threads that live on after a read hold nothing.
CACTI_API int cacti_hip_read_i32(const void *dev, int32_t *value, void *stream)
{
    CACTI_REQUIRE(dev && value && aligned(dev, 16), CACTI_E_INVALID, "read_i32: null or misaligned pointer");
    Staging s;
    if (!staging_take(&s, kWordBytes)) {
        CACTI_HIP(hipMemcpyAsync(value, dev, sizeof(*value), hipMemcpyDeviceToHost, (hipStream_t)stream));
        CACTI_HIP(hipStreamSynchronize((hipStream_t)stream));
        return 0;
    }
    const HostRegion r = {dev, s.data(), sizeof(*value)};
    const int rc = gather_to_host(s, &r, 1, (hipStream_t)stream);
    if (!rc) memcpy(value, s.data(), sizeof(*value));
    staging_give_back(&s);
    return rc;
}

CACTI_API int cacti_hip_pinned_bytes(size_t *held, size_t *kept)
{
    CACTI_REQUIRE(held && kept, CACTI_E_INVALID, "pinned_bytes: null out pointer");
    std::lock_guard<std::mutex> lock(g_mutex);
    *held = g_pinned.load();
    *kept = 0;
    for (const Kept &k : g_kept) *kept += k.bytes * (size_t)k.n;
    return 0;
}
