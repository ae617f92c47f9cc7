// The host's side of a large read: pieces of a window are copied on as they arrive, by a few threads.  (No device code and
// no HIP call: the caller says how to wait for a piece.)
#pragma once
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <mutex>
#include <thread>

namespace cacti {

constexpr int kCopyThreads = 4;

// The first failure of any of the threads, with its text: error texts belong to the thread that failed.
struct ChunkError {
    int rc = 0;
    char text[512] = "";
};

// Copies `bytes` from src to dst in pieces of `chunk`, on this thread and up to threads - 1 others (start() runs first on
// each of those).  Piece i is copied once wait(i) has returned 0; after any other status no further piece is begun, and
// message() is asked, on the thread it came up on, for its text.
template <class Start, class Wait, class Message>
ChunkError copy_chunks(char *dst, const char *src, size_t bytes, size_t chunk, int threads, Start start, Wait wait, Message message)
{
    const int chunks = (int)((bytes + chunk - 1) / chunk);
    std::atomic<int> next{0};
    std::atomic<bool> failed{false};
    std::mutex mutex;
    ChunkError error;
    auto work = [&]() {
        for (int i; !failed.load() && (i = next.fetch_add(1)) < chunks;) {
            const int rc = wait(i);
            if (rc == 0) {
                memcpy(dst + (size_t)i * chunk, src + (size_t)i * chunk, std::min(chunk, bytes - (size_t)i * chunk));
                continue;
            }
            std::lock_guard<std::mutex> lock(mutex);
            if (!failed.exchange(true)) {
                error.rc = rc;
                snprintf(error.text, sizeof(error.text), "%s", message());
            }
        }
    };
    std::thread th[kCopyThreads];
    try {
        for (int t = 1; t < std::min(threads, kCopyThreads); t++)
            th[t] = std::thread([&]() {
                start();
                work();
            });
    } catch (const std::exception &) {
        // no more threads (or memory for one) to be had: those that started and this one take the pieces
    }
    work();
    for (std::thread &t : th)
        if (t.joinable()) t.join();
    return error;
}

}  // namespace cacti
