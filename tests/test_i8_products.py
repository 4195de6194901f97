"""int8 MATMUL at any alignment: the edges of the stages, tiles and register sets of product_i8.hip, against whole-number sums."""
import numpy as np
import pytest

from test_ragged_contractions import abi, hb, i8, run, scale  # noqa: F401
from hip_util import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

# batch, m, k, n
EDGES = [
    (1, 1, 16, 17), (2, 3, 255, 19), (1, 5, 256, 33), (1, 33, 257, 31), (3, 4, 1023, 7), (1, 2, 1281, 15), (1, 1, 2817, 45),
    (2, 37, 1537, 29),                       # 32 x 32: one stage, its edges, every remainder of the four register sets
    (70, 65, 129, 63), (33, 130, 257, 95), (40, 64, 769, 61), (40, 63, 513, 127),  # 64 x 64
    (1, 2050, 130, 2049), (1, 2049, 385, 2047), (70, 257, 128, 129),               # 128 x 128
]


@pytest.mark.parametrize("b_rows", [False, True], ids=["kmajor", "rows"])
@pytest.mark.parametrize("case", EDGES, ids=["x".join(map(str, c)) for c in EDGES])
def test_product_edges(run, case, b_rows):  # noqa: F811
    nb, m, k, n = case
    rng = np.random.default_rng(sum(case))
    a, b = i8(rng, (nb, m, k)), i8(rng, (nb, k, n))
    sums = np.stack([(x.astype(np.float64) - 3) @ (y.astype(np.float64) + 5) for x, y in zip(a, b)]).astype(np.int64)
    np.testing.assert_array_equal(run.matmul(a, b, abi.I32, 3, -5, b_rows=b_rows), sums.astype(np.int32))
    mult, shift = scale(rng, 1, k)
    rattr = abi.rescale_attr(0, -2, True, False, False)
    out = run.matmul(a, b, abi.I8, 3, -5, epilogue=(mult, shift, rattr, None), b_rows=b_rows)
    exp = np.clip(((sums * int(mult[0]) + (1 << (int(shift[0]) - 1))) >> int(shift[0])) - 2, -128, 127)
    np.testing.assert_array_equal(out, exp.astype(np.int8))
