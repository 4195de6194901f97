"""fp16 products over row-wise weights at the edges of every tile of the direct-to-LDS loop, against float64 sums."""
import numpy as np
import pytest

from hip_util import gpu_available
from test_float_contractions import run  # noqa: F401

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

CASES = [
    # m, k, n
    (65, 64, 72), (1, 128, 8), (130, 320, 200), (63, 96, 136),        # at most two tiles of 32 x 32 per unit: the kernel of few tiles
    (1005, 320, 712), (999, 288, 600),                                 # 64 x 64: steps of 64 halfs, of 32
    (3900, 256, 2296), (4096, 288, 2304),                              # 256 x 192
    (4000, 256, 3080),                                                 # 256 x 256
    (1700, 832, 1496), (1665, 1024, 1544),                             # 128 x 128, steps of 64
    (1700, 800, 1496), (5000, 64, 1400),                               # 128 x 128, steps of 32
]


@pytest.mark.parametrize("case", CASES, ids=["x".join(map(str, c)) for c in CASES])
def test_row_wise_tiles(run, case):  # noqa: F811
    m, k, n = case
    rng = np.random.default_rng(sum(case))
    a = rng.standard_normal((1, m, k)).astype(np.float16)
    b = rng.standard_normal((1, k, n)).astype(np.float16)
    bias = rng.standard_normal((1, 1, n)).astype(np.float32)
    want = np.matmul(a.astype(np.float32), b.astype(np.float32)) + bias
    got = run.matmul_bias_cast(a, b, bias, b_rows=True)
    np.testing.assert_allclose(got.astype(np.float32), want, rtol=1e-3, atol=1e-5 * k)
    res = rng.standard_normal((1, m, n)).astype(np.float16)
    np.testing.assert_array_equal(run.matmul_bias_cast_add(a, b, bias, res, b_rows=True), got + res)
    if n % 3 == 0 and n // 3 % 8 == 0:
        parts = run.matmul_bias_cast_group(a, np.split(b, 3, 2), np.split(bias, 3, 2), b_rows=True)
        np.testing.assert_array_equal(np.concatenate(parts, 2), got)
