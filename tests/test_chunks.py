"""The host's side of a large read (csrc/chunks.h): pieces copied on by several threads, and what a failure of one of them
leaves behind.  The header has no device code; it is compiled into a small program here and run on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <stdlib.h>

#include <vector>

#include "chunks.h"

using namespace cacti;

static thread_local char t_error[64] = "old";

#define CHECK(x) do { if (!(x)) { printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

int main()
{
    const size_t bytes = 10 * 64 + 17, chunk = 64;
    std::vector<char> src(bytes), dst(bytes);
    for (size_t i = 0; i < bytes; i++) src[i] = (char)rand();
    const std::thread::id here = std::this_thread::get_id();
    for (int threads : {1, 2, 4, 9}) {
        // every piece once, also the short last one
        std::fill(dst.begin(), dst.end(), 0);
        std::atomic<int> waits{0}, starts{0};
        ChunkError e = copy_chunks(dst.data(), src.data(), bytes, chunk, threads, [&]() { starts++; }, [&](int) { waits++; return 0; },
                                   []() { return t_error; });
        CHECK(e.rc == 0 && dst == src && waits == 11 && starts == std::min(threads, kCopyThreads) - 1);
    }
    // Piece 1 fails on a helper thread, piece 0 on this one is only there after that: status and text of the failure come
    // back, this thread's own text stays, and the other pieces are left.
    for (int round = 0; round < 50; round++) {
        std::fill(dst.begin(), dst.end(), 0);
        std::atomic<bool> failing{false};
        std::atomic<int> waits{0};
        ChunkError e = copy_chunks(
            dst.data(), src.data(), bytes, chunk, 2, []() {},
            [&](int) {
                waits++;
                if (std::this_thread::get_id() == here) {
                    while (!failing.load()) std::this_thread::yield();
                    return 0;
                }
                snprintf(t_error, sizeof(t_error), "piece lost, round %d", round);
                failing.store(true);
                return -5;
            },
            []() { return t_error; });
        char want[64];
        snprintf(want, sizeof(want), "piece lost, round %d", round);
        CHECK(e.rc == -5 && !strcmp(e.text, want) && !strcmp(t_error, "old"));
        CHECK(waits <= 11);
    }
    return 0;
}
"""


def test_chunks_and_the_text_of_a_failure(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-Wall", "-Werror", "-pthread",
                           "-I" + os.path.join(ROOT, "cacti_amd", "csrc"), str(src), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
