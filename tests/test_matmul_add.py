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


@pytest.mark.parametrize("b_rows", [False, True], ids=["k_major", "row_wise"])
@pytest.mark.parametrize("case", [(1, 3900, 4096, 4088, 4088), (3, 2048, 3072, 2040, 1), (1, 4096, 2048, 4096, 4096)])
def test_large_fp16_products_with_a_row(run, case, b_rows):  # noqa: F811
    """Both sides of the line between one launch and the product with the ADD behind it, against the operators one by one: the
    same sums in fp32 up to the order of their additions, and every row and column where it belongs."""
    nb, m, k, n, row = case
    rng = np.random.default_rng(sum(case))
    a, b = (rng.standard_normal((nb, i, j), dtype=np.float32).astype(np.float16) for i, j in ((m, k), (n, k) if b_rows else (k, n)))
    bias = rng.standard_normal((1, 1, row)).astype(np.float32)
    ta, tb, tr = run.put(a), run.put(b), run.put(bias)
    to, tp, ts = (run.new(abi.F32, (nb, m, n)) for _ in range(3))
    view = abi.make_tensor(tb.ptr, abi.F16, (nb, k, n), [n * k * 2, 2, k * 2]) if b_rows else tb.view
    attr = abi.MatmulAttr(0, 0)
    run.dev.op("matmul_add", to.ref, ta.ref, C.byref(view), C.byref(attr), tr.ref)
    run.dev.op("matmul", tp.ref, ta.ref, C.byref(view), C.byref(attr))
    run.dev.op("elementwise_binary", abi.BIN["ADD"], ts.ref, tp.ref, tr.ref, abi.NAN_PROPAGATE)
    got, want = to.download(), ts.download()
    run.done()
    # two fp32 sums of k products of a size around one: each off by at most some sqrt(k) 2^-24 of their size
    np.testing.assert_allclose(got, want, rtol=0, atol=8 * k * 2.0 ** -24)
    some = rng.integers(0, m, 4)
    exact = a[0, some].astype(np.float64) @ (b[0].T if b_rows else b[0]).astype(np.float64) + bias[0]
    np.testing.assert_allclose(got[0, some], exact, rtol=0, atol=8 * k * 2.0 ** -24)
