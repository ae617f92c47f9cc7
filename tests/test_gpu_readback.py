"""Read-backs: page-locked memory the library holds for them, and readers that do not get in each other's way (MI355X)."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def pinned():
    from cacti_amd import ffi
    held, kept = C.c_size_t(), C.c_size_t()
    ffi.call("cacti_hip_pinned_bytes", C.byref(held), C.byref(kept))
    return held.value, kept.value


def test_reading_a_word_holds_no_memory_per_thread():
    """Threads that stay alive after a read of one word hold nothing, and what is kept for later reads stays small however
    many threads read at once."""
    import torch
    from cacti_amd import ffi
    words = torch.arange(0, 48 * 4, 4, dtype=torch.int32, device="cuda").view(48, 1).repeat(1, 4).contiguous()
    torch.cuda.synchronize()
    before = pinned()
    got, read, done = [None] * 48, threading.Barrier(49, timeout=60), threading.Barrier(49, timeout=60)

    def work(i):
        v = C.c_int32(-1)
        ffi.call("cacti_hip_read_i32", words[i].data_ptr(), C.byref(v), None)
        got[i] = v.value
        read.wait()
        done.wait()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(48)]
    for t in threads:
        t.start()
    read.wait()                                            # all have read, all are alive
    after = pinned()
    done.wait()
    for t in threads:
        t.join()
    assert got == [4 * i for i in range(48)]
    assert after[0] - before[0] <= 16 * 8192 and after[0] - after[1] == before[0] - before[1]
