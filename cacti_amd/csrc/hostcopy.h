#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace cacti {

// A device region (16-byte aligned; the whole last 16 bytes are readable) and where it goes in page-locked memory.
struct HostRegion {
    const void *src;
    void *dst;
    size_t bytes;
};
constexpr int kMaxRegions = 8;

// Page-locked memory regions are gathered into, with the words their arrival is announced in.  One gather at a time.
struct Staging {
    char *base = nullptr;
    size_t bytes = 0;
    unsigned epoch = 0;
    int dev = 0;                               // the device that was current when it was page-locked
    unsigned resets = 0;                       // and how often that had been reset
    bool lost = false;                         // a failed read may still be writing it
    char *data() const { return base + kFlagBytes; }
    size_t room() const { return bytes - kFlagBytes; }
    static constexpr size_t kFlagBytes = 4096;
};
constexpr size_t kStagingBytes = 4u << 20;     // of a context
constexpr size_t kWordBytes = 8u << 10;        // of a call that reads one word
constexpr size_t kWindowBytes = Staging::kFlagBytes + (16u << 20);   // of a large read: a window of it at a time
// n <= kMaxRegions regions, in one launch on `st`, to places in s.data(); returns when they are there.  The launch comes
// behind all work queued on `st`, so this waits for it like a stream synchronisation.
int gather_to_host(Staging &s, const HostRegion *r, int n, hipStream_t st);
// one region of any size to pageable memory, likewise, and (not null) a word of device memory with it: up to kOwnRead bytes
// through `own`, the caller's, which no other reader waits for or takes; beyond through a borrowed window.  Readers on
// other threads and streams go on meanwhile.
int read_large(Staging &own, void *dst, const void *src, size_t bytes, const int *word, int *word_dst, hipStream_t st);
constexpr size_t kLargeRead = 192u << 10;      // from here on it is the better one where there is something else to gather,
constexpr size_t kLargeAlone = 96u << 10;      // and from here on where there is not
constexpr size_t kOwnRead = 512u << 10;
static_assert(kOwnRead <= kStagingBytes - Staging::kFlagBytes, "a context's buffer holds it");
// n regions of `bytes` (a multiple of 16), 16-byte aligned, set to zero
int zero_regions(void *const *ptrs, int n, size_t bytes, hipStream_t st);

// A buffer of one of the sizes above, for the current device.  A few of each size that were given back are kept for later
// takers (page-locking costs hundreds of microseconds).
bool staging_take(Staging *s, size_t bytes);
void staging_give_back(Staging *s);
// Before a reset of the device, which deletes its page-locked memory too: frees what is kept, and what is in use then is
// not kept later.
void staging_release(int dev);

}  // namespace cacti
