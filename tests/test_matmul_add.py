"""MATMUL + ADD of a row in one launch, against float64 sums."""
import ctypes as C

import numpy as np
import pytest

from hip_util import gpu_available
from test_float_contractions import abi, floats, run, values  # noqa: F401

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.mark.parametrize("dt", [abi.F16, abi.BF16, abi.F32], ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", [(1, 1, 16, 10, 10), (1, 33, 100, 257, 1), (3, 5, 64, 31, 31), (1, 70, 300, 1000, 1000)])
def test_matmul_add(run, case, dt):  # noqa: F811
    nb, m, k, n, row = case
    rng = np.random.default_rng(sum(case))
    a, b = values(rng, (nb, m, k), dt), values(rng, (nb, k, n), dt)
    bias = rng.standard_normal((1, 1, row)).astype(np.float32)
    ta, tb, tr, to = run.put(a, dt), run.put(b, dt), run.put(bias), run.new(abi.F32, (nb, m, n))
    attr = abi.MatmulAttr(0, 0)
    assert run.dev.lib.mlel_hip_matmul_add_in_kernel(to.ref, ta.ref, tb.ref, C.byref(attr), tr.ref) == 1
    run.dev.op("matmul_add", to.ref, ta.ref, tb.ref, C.byref(attr), tr.ref)
    got = to.download()
    run.done()
    want = np.matmul(floats(a).astype(np.float64), floats(b).astype(np.float64)) + bias
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-6 * k)
    assert run.dev.lib.mlel_hip_matmul_add_in_kernel(to.ref, ta.ref, tb.ref, C.byref(abi.MatmulAttr(1, 0)), tr.ref) == 0
