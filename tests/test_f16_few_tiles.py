"""fp16 products of few tiles (gemm_f16_few_kernel) and around its borders: every layout and form of a product gives the bits of
the plain MATMUL followed by the operators, and that is within the rounding of fp32 sums of the exact product."""
import ctypes as C
import importlib

import numpy as np
import pytest

from hip_util import gpu_available
from test_float_contractions import run  # noqa: F401

abi = importlib.import_module("ai-ml-emulation-layer-for-vulkan_amd.abi")

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

CASES = [
    # batches, m, k, n
    (1, 1, 32, 8), (3, 33, 64, 40), (1, 31, 96, 72), (2, 32, 128, 32), (1, 64, 160, 200), (1, 65, 544, 24),
    (1, 100, 1536, 264),                       # whole stages, one tile per unit
    (1, 200, 416, 1192), (5, 197, 64, 200),    # two tiles per unit
    (1, 600, 288, 1000),                       # K-major: three tiles per unit; row-wise: 64 x 64, steps of 32
    (1, 1000, 320, 712),                       # row-wise: 64 x 64, steps of 64; K-major: three tiles per unit
    # K-major products that keep to gemm_f16.hip's tiles: few rows, few columns, half of 128 columns, a round of 128 x 128, a little more
    (9, 3, 32, 2048), (13, 1300, 96, 16), (1, 705, 288, 1032), (1, 1300, 768, 1920), (1, 2500, 160, 1664),
    (1, 1030, 1088, 1048),                     # K-major MATMUL of long rows without shared K
    (1, 2050, 320, 2056),                      # K-major: 128 x 128
]


def data(case):
    nb, m, k, n = case
    rng = np.random.default_rng(sum(case))
    a, b = rng.standard_normal((nb, m, k)).astype(np.float16), rng.standard_normal((nb, k, n)).astype(np.float16)
    return a, b, rng.standard_normal((1, 1, n)).astype(np.float32), rng.standard_normal((nb, m, n)).astype(np.float16)


@pytest.mark.parametrize("case", CASES, ids=["x".join(map(str, c)) for c in CASES])
def test_every_form_gives_the_same_bits(run, case):  # noqa: F811
    a, b, bias, res = data(case)
    plain = run.matmul(a, b, abi.F32)
    exact = np.matmul(a.astype(np.float64), b.astype(np.float64))
    size = np.matmul(np.abs(a.astype(np.float64)), np.abs(b.astype(np.float64)))
    # K - 1 additions of exact products, each rounded once (a matrix instruction adds sixteen at a time)
    assert np.all(np.abs(plain - exact) <= case[2] * 2.0 ** -24 * size)
    np.testing.assert_array_equal(run.matmul(a, b, abi.F32, b_rows=True), plain)
    want = (plain + bias).astype(np.float16)
    for rows in (False, True):
        np.testing.assert_array_equal(run.matmul_bias_cast(a, b, bias, b_rows=rows), want)
        np.testing.assert_array_equal(run.matmul_bias_cast_add(a, b, bias, res, b_rows=rows), want + res)
    if case[0] == 1 and case[3] % 24 == 0:
        parts = run.matmul_bias_cast_group(a, np.split(b, 3, 2), np.split(bias, 3, 2), b_rows=True)
        np.testing.assert_array_equal(np.concatenate(parts, 2), want)


@pytest.mark.parametrize("transposing", [False, True], ids=["split", "transposing"])
@pytest.mark.parametrize("k", [40, 96])
def test_views_of_few_tiles(run, k, transposing):  # noqa: F811
    """The result through a view [2, 1, 3, 16, 5, 8]: heads side by side, or with the rows innermost."""
    rng = np.random.default_rng(k)
    nb, m, n = 2, 48, 40
    a, b = rng.standard_normal((nb, m, k)).astype(np.float16), rng.standard_normal((nb, k, n)).astype(np.float16)
    bias = rng.standard_normal((1, 1, n)).astype(np.float32)
    want = run.matmul_bias_cast(a, b, bias)
    dims = (2, 1, 3, 16, 5, 8)
    order = (0, 4, 5, 1, 2, 3) if transposing else (0, 4, 1, 2, 3, 5)  # of the six axes in memory
    strides, step = [0] * 6, 2
    for axis in reversed(order):
        strides[axis], step = step, step * dims[axis]
    rows = k % 32 == 0
    es = 2
    ta, tbias = run.put(a), run.put(bias)
    tb = run.put(np.ascontiguousarray(np.transpose(b, (0, 2, 1))) if rows else b)
    bv = abi.make_tensor(tb.ptr, abi.F16, (nb, k, n), (n * k * es, es, k * es)) if rows else tb.view
    to = run.new(abi.F16, (nb * m * n,))
    view = abi.make_tensor(to.ptr, abi.F16, dims, strides)
    run.dev.op("matmul_bias_cast", C.byref(view), ta.ref, C.byref(bv), tbias.ref, C.byref(abi.MatmulAttr(0, 0)))
    got = to.download().reshape([dims[x] for x in order])
    run.done()
    np.testing.assert_array_equal(got, want.reshape(dims).transpose(order))
