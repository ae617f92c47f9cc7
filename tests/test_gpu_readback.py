"""Read-backs: page-locked memory the library holds for them, and readers that do not get in each other's way (MI355X)."""
import ctypes as C
import os
import subprocess
import sys
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def pinned():
    from cacti_amd import ffi
    held, kept = C.c_size_t(), C.c_size_t()
    ffi.call("cacti_hip_pinned_bytes", C.byref(held), C.byref(kept))
    return held.value, kept.value


def test_reading_a_word_holds_no_memory_per_thread():
    """Threads that stay alive after a read of one word hold nothing, and what is kept for later reads stays small however
    many threads read at once."""
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


SMALL = dict(S=32, D=256, H=4, F=512, L=1, eps=1e-6)


def model(V=4096, pagelocked=True):
    from cacti_amd.runtime import Ctx, Llama
    ctx = Ctx(0, 256 << 20, pagelocked)
    m = Llama(ctx, SMALL["S"], SMALL["D"], SMALL["H"], SMALL["D"] // SMALL["H"], SMALL["F"], V, SMALL["L"], SMALL["eps"])
    r = np.random.default_rng(3)
    for i, (name, shape) in enumerate(m.params):
        m.put_param(i, (r.standard_normal(shape) * 0.05).astype(np.float16))
    tok = r.integers(0, V, SMALL["S"]).astype(np.uint16)
    m.step(tok, tok, np.full(SMALL["S"], 8.0, np.float32))
    return ctx, m


def busy(stream, ms):
    """Keeps a stream busy for about that long (a kernel that counts clock cycles)."""
    st = torch.cuda.ExternalStream(stream, device="cuda:0")
    with torch.cuda.stream(st):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        torch.cuda._sleep(1000)
        a.record()
        torch.cuda._sleep(1000000)
        b.record()
        b.synchronize()
        torch.cuda._sleep(int(min(ms / a.elapsed_time(b), 2000) * 1000000))


def concurrent_reads():
    from cacti_amd import ffi
    torch.cuda.init()
    # (no streams for spilling: two streams and the null stream are fewer than the hardware queues, so none shares one)
    (ctx_a, a), (ctx_b, b) = model(pagelocked=False), model(pagelocked=False)
    i = [n for n, _ in a.params].index("lm_head")
    want = a.grad(i)
    assert want.nbytes >= 2 << 20 and np.array_equal(want, b.grad(i))
    got = {}

    def slow():
        got["a"] = a.grad(i)

    busy(ffi.lib().cacti_ctx_stream(ctx_a._c), 1500.0)
    t = threading.Thread(target=slow)
    t.start()
    t.join(0.1)                                            # it is inside its read by now
    got["b"] = b.grad(i)
    first = t.is_alive()
    t.join()
    assert np.array_equal(got["a"], want) and np.array_equal(got["b"], want)
    for x in (a, b, ctx_a, ctx_b):
        x.close()
    print("the other context's read was first:", first)


def child(code):
    """Runs in a process of its own: with its own hardware queues, and its own device state."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", "import sys; sys.path.insert(0, %r); import torch; torch.cuda.init()\n%s" % (root, code)],
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr[-2000:]
    return r.stdout


def test_a_large_read_does_not_wait_for_another_contexts_stream():
    """One context's large read waits for what is queued on its stream; a read of another context, on another thread, is
    through before that."""
    assert "first: True" in child("from tests.test_gpu_readback import concurrent_reads; concurrent_reads()")


def test_reads_of_some_hundred_kb_at_once_page_lock_nothing():
    """Three contexts read a gradient of 300 KB at the same time, each waiting for what is queued on its own stream: each
    goes through the buffer its context has anyway."""
    from cacti_amd import ffi
    contexts = [model(V=600, pagelocked=False) for _ in range(3)]
    i = [n for n, _ in contexts[0][1].params].index("lm_head")
    want = contexts[0][1].grad(i)
    assert 192 << 10 < want.nbytes < 512 << 10
    got = [None] * 3

    def read(j):
        got[j] = contexts[j][1].grad(i)

    torch.cuda.synchronize()
    before = pinned()
    for ctx, _ in contexts:
        busy(ffi.lib().cacti_ctx_stream(ctx._c), 400.0)
    threads = [threading.Thread(target=read, args=(j,)) for j in range(3)]
    for t in threads:
        t.start()
    threads[0].join(0.1)                                   # all three are inside their reads by now
    during = pinned()
    for t in threads:
        t.join()
    for g in got:
        assert np.array_equal(g, want)
    assert during[0] == pinned()[0] == before[0]
    for ctx, m in contexts:
        m.close(); ctx.close()


def test_a_context_reads_large_and_small_through_one_buffer():
    """Reads in chunks (300 KB, with the status word behind it) and in one gather, in turn: the words that announce them
    share their place in the context's buffer."""
    ctx, m = model(V=600)
    names = [n for n, _ in m.params]
    big, small = names.index("lm_head"), names.index("head_norm")
    want = None
    r = np.random.default_rng(4)
    tok = r.integers(0, 600, SMALL["S"]).astype(np.uint16)
    for _ in range(40):
        m.step(tok, tok, np.full(SMALL["S"], 8.0, np.float32))
        now = m.grad(big), m.grad(small)
        want = want or now
        for _ in range(3):
            again = m.grad(small), m.grad(big)
            assert np.array_equal(again[0], now[1]) and np.array_equal(again[1], now[0])
        assert np.array_equal(now[0], want[0]) and np.array_equal(now[1], want[1])
    m.close(); ctx.close()


@pytest.mark.parametrize("V,D", [(20000, 1024), (8200, 1032), (24, 264)])
def test_reads_of_several_windows_come_back_whole(V, D):
    """41 MB in three windows of 16 MiB; 16.9 MB, a window and a few pieces, the last of them short; 13 KB in one gather.
    Right behind an update on the device, so that the bytes are not the host's own copy."""
    from cacti_amd.runtime import Ctx, Llama
    ctx = Ctx(0, 1 << 30, True)
    m = Llama(ctx, 16, D, 4, D // 4, 64, V, 0, 1e-6)
    r = np.random.default_rng(V)
    for i, (name, shape) in enumerate(m.params):
        m.put_param(i, (r.standard_normal(shape) * 0.05).astype(np.float16))
    tok = r.integers(0, V, 16).astype(np.uint16)
    m.adamw_init()
    m.step(tok, tok, np.full(16, 8.0, np.float32))
    m.adamw_step(1, lr=1e-2)
    for i, (name, shape) in enumerate(m.params):
        # the f16 parameter is the rounded master, which comes back through another read of twice the bytes
        got, master = m.param(i), m.adamw_state(i, "master")
        assert np.array_equal(got.view(np.uint16), master.astype(np.float16).view(np.uint16)), name
        assert np.isfinite(master).all() and len(np.unique(got.view(np.uint16))) > min(got.size, 100) // 4
    m.close(); ctx.close()


def test_a_device_reset_leaves_no_page_locked_buffer():
    """The buffers kept for later contexts go before the reset that would delete them under the library (a child process:
    the reset takes everything on the device with it)."""
    assert "released" in child(
        "from cacti_amd import ffi\n"
        "from tests.test_gpu_readback import model, pinned\n"
        "ctx, m = model()\n"
        "m.grads()\n"
        "m.close(); ctx.close()\n"
        "held, kept = pinned()\n"
        "assert held == kept >= (16 << 20), (held, kept)\n"
        "ffi.call('cacti_hip_primary_ctx_reset', 0)\n"
        "assert pinned() == (0, 0), pinned()\n"
        "print('released')\n")
