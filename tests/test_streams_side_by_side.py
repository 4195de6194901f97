"""The streams that a program makes first run side by side: the library takes no turn when the runtime deals its hardware queues to
streams.  In a process of its own, since the streams of the tests before have taken theirs."""
import pathlib
import subprocess
import sys

import pytest

from hip_util import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

PROGRAM = """
import ctypes as C, importlib, time
import numpy as np
abi = importlib.import_module("ai-ml-emulation-layer-for-vulkan_amd.abi")
hb = importlib.import_module("ai-ml-emulation-layer-for-vulkan_amd.hip_backend")
dev = hb.Device(0)
a, b = dev.from_numpy(np.ones((1, 16, 65536), np.float32)), dev.from_numpy(np.ones((1, 65536, 16), np.float32))
streams = [dev.new_stream() for _ in range(3)]
outs = [dev.tensor(abi.F32, (1, 16, 16)) for _ in streams]

def time_on(which):
    best = 1e9
    for _ in range(5):
        dev._check(dev.lib.mlel_hip_sync(dev.ctx, None))
        t = time.perf_counter()
        for k in range(20):
            i = which[k % len(which)]
            dev.stream = streams[i]
            dev.op("matmul", outs[i].ref, a.ref, b.ref, C.byref(abi.MatmulAttr(0, 0)))
        dev._check(dev.lib.mlel_hip_sync(dev.ctx, None))
        best = min(best, time.perf_counter() - t)
    return best

time_on([0, 1, 2])
print(time_on([0]), time_on([0, 1]), time_on([1, 2]))
assert all((t.download() == 65536).all() for t in outs)
"""


def test_two_streams_run_one_block_each_at_the_same_time():
    """A product of one tile leaves the chip to the other stream's: two streams take half the time of one, where they share a queue
    all of it."""
    root = pathlib.Path(__file__).parents[1]
    out = subprocess.run([sys.executable, "-c", PROGRAM], cwd=root, capture_output=True, text=True, timeout=90)
    assert out.returncode == 0, out.stderr
    one, first, second = map(float, out.stdout.split()[-3:])
    assert first < 0.75 * one and second < 0.75 * one, (one, first, second)
