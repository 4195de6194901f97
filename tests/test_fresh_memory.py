"""Memory that was just allocated is zero and stays what a stream of the library writes there first."""
import ctypes as C
import threading

import numpy as np
import pytest

from hip_util import gpu_available, hb

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.mark.parametrize("mib", [1, 64, 1024])
def test_a_copy_onto_fresh_memory_is_not_overtaken_by_its_clearing(mib):
    """The clearing of an allocation has ended when the call returns: a copy on another stream keeps its bytes, at the end of the
    allocation, which is cleared last."""
    dev = hb.Device(0)
    dev.stream = stream = dev.new_stream()
    size, tail = mib << 20, np.random.default_rng(mib).integers(-128, 127, 1 << 16).astype(np.int8)
    for _ in range(3):
        ptr = dev.alloc(size)
        dev.h2d(ptr + size - tail.nbytes, tail.ctypes.data, tail.nbytes)
        got, head = np.empty_like(tail), np.ones(4096, np.int8)
        dev.d2h(head.ctypes.data, ptr, head.nbytes)
        dev.d2h(got.ctypes.data, ptr + size - tail.nbytes, got.nbytes)
        assert not head.any()
        np.testing.assert_array_equal(got, tail)
        dev.free(ptr)
    dev.stream = None
    dev.free_stream(stream)
    dev.close()


def test_small_allocations_are_apart_zero_and_taken_again():
    """Allocations of every small size, some written and freed in between: none overlaps another, all are zero when handed out."""
    dev = hb.Device(0)
    rng, live = np.random.default_rng(3), []
    for i in range(200):
        size = int(rng.choice([1, 16, 4096, 4097, 9000, 16384, 40000, 65536, 65537]))
        ptr, got, sevens = dev.alloc(size), np.ones(size, np.int8), np.full(size, 7, np.int8)
        dev.d2h(got.ctypes.data, ptr, size)
        assert ptr % 256 == 0 and not got.any()
        assert all(ptr + size <= p or p + n <= ptr for p, n in live)
        dev.h2d(ptr, sevens.ctypes.data, size)
        live.append((ptr, size))
        if i % 3 == 2:
            dev.free(live.pop(int(rng.integers(len(live))))[0])
    for ptr, _ in live:
        dev.free(ptr)
    dev.close()


def test_a_capture_refuses_every_allocation_also_of_what_lies_ready():
    """Small allocations are made ahead, and a thread that captures is refused them as it is refused a large one; outside the capture
    they are zero again."""
    dev = hb.Device(0)
    live = [dev.alloc(size) for size in (16, 16, 65536)]  # from now on others lie ready
    refused = []

    def capture():  # on a thread of its own: the runtime keeps a thread's last error, and a stream whose capture has failed
        stream, exe = dev.new_stream(), C.c_void_p()
        dev._check(dev.lib.mlel_hip_capture_begin(dev.ctx, stream))
        for size in (16, 65536, 1 << 20):
            try:
                dev.alloc(size)
            except hb.MlelError as e:
                refused.append(str(e))
        dev.lib.mlel_hip_capture_end(dev.ctx, stream, C.byref(exe))

    thread = threading.Thread(target=capture)
    thread.start()
    thread.join()
    assert len(refused) == 3 and all("hipMalloc" in text for text in refused)
    for size in (16, 65536, 1 << 20) * 10:
        ptr, got = dev.alloc(size), np.ones(size, np.int8)
        dev.d2h(got.ctypes.data, ptr, size)
        assert not got.any()
        live.append(ptr)
    assert len(set(live)) == len(live)
    for ptr in live:
        dev.free(ptr)
    dev.close()


def test_threads_share_the_allocations_made_ahead():
    """Four threads allocate from one device at a time: zero, none overlapping another, each keeping what was written there."""
    dev = hb.Device(0)
    taken, wrong = [[] for _ in range(4)], []

    def work(t):
        rng = np.random.default_rng(t)
        try:
            for _ in range(100):
                size = int(rng.choice([1, 4096, 4097, 16384, 65536]))
                ptr, got, mark = dev.alloc(size), np.ones(size, np.int8), np.full(size, t + 1, np.int8)
                dev.d2h(got.ctypes.data, ptr, size)
                if got.any():
                    wrong.append((t, ptr, size))
                dev.h2d(ptr, mark.ctypes.data, size)
                taken[t].append((ptr, size))
        except Exception as e:  # noqa: BLE001
            wrong.append(e)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    blocks = sorted(b for per in taken for b in per)
    assert all(p + n <= q for (p, n), (q, _) in zip(blocks, blocks[1:]))
    for t, per in enumerate(taken):
        for ptr, size in per:
            got = np.zeros(size, np.int8)
            dev.d2h(got.ctypes.data, ptr, size)
            assert (got == t + 1).all()
            dev.free(ptr)
    dev.close()
