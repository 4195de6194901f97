"""CONV2D over floating-point tensors whose weights hold infinities and NaN: a tap outside the image contributes nothing
(conv2d.comp:40-116), so what such a weight does to the inside of an image must not reach the positions at its border."""
import zlib

import numpy as np
import pytest

from hip_util import gpu_available
from test_float_contractions import STEP, TYPES, abi, floats, run, values  # noqa: F401

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

CASES = [
    # n, h, w, ic, oc, kernel, stride, dilation, pad
    (2, 7, 9, 16, 24, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),      # aligned pieces, tiles of 16 x 16
    (1, 40, 41, 16, 64, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),    # 32 x 32
    (1, 64, 130, 8, 64, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),    # 64 x 64
    (1, 256, 257, 8, 72, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),   # 128 x 128
    (2, 13, 12, 3, 20, (3, 3), (2, 2), (1, 1), (0, 1, 1, 1)),     # kernel rows from any address
    (1, 64, 130, 3, 61, (5, 3), (1, 1), (1, 1), (2, 2, 1, 1)),
    (1, 9, 11, 5, 7, (3, 3), (1, 1), (2, 2), (2, 2, 2, 2)),       # element by element
    (1, 12, 10, 16, 9, (3, 3), (2, 1), (2, 2), (0, 3, 2, 2)),
    (1, 3, 3, 8, 5, (3, 3), (1, 1), (1, 1), (4, 4, 4, 4)),        # positions that meet no pixel at all
]


@pytest.mark.parametrize("dt", TYPES, ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", CASES, ids=["_".join(map(str, c[1:5] + c[5] + c[7])) for c in CASES])
def test_weights_that_are_not_finite(run, oracle, case, dt):  # noqa: F811
    n, h, w, ic, oc, (kh, kw), (sy, sx), (dy, dx), pad = case
    rng = np.random.default_rng(zlib.crc32(repr(case).encode()))
    x, wt = values(rng, (n, h, w, ic), dt), values(rng, (oc, kh, kw, ic), dt, (kh * kw * ic) ** -0.5)
    b = values(rng, (oc,), dt)
    special = np.array([0x7f80, 0xff80, 0x7fc0], np.uint16) if dt == abi.BF16 else np.array([np.inf, -np.inf, np.nan], wt.dtype)
    for c in range(oc):  # one tap of every channel, each tap in turn; every fourth channel stays finite
        if c % 4 < 3:
            wt[c, c % kh, (c // kh) % kw, c % ic] = special[c % 4]
    shape = (n, (h + pad[0] + pad[1] - (kh - 1) * dy - 1) // sy + 1, (w + pad[2] + pad[3] - (kw - 1) * dx - 1) // sx + 1, oc)
    attr = abi.conv2d_attr(pad, (sy, sx), (dy, dx), acc_type=abi.ACC_F32)
    got = floats(run.conv2d(x, wt, b, shape, dt, attr))
    want = floats(oracle.conv2d(x, wt, b, shape, dt, attr))
    border = ~np.isfinite(want)
    assert border.any() and not border.all()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fine = np.isfinite(want)
    np.testing.assert_allclose(got[fine], want[fine], rtol=1.01 * STEP[dt], atol=2e-5)


@pytest.mark.parametrize("dt", TYPES, ids=["f16", "bf16", "f32"])
def test_images_that_are_not_finite(run, oracle, dt):  # noqa: F811
    """A NaN and an infinity in the image: their neighbourhoods only, at the border as inside."""
    rng = np.random.default_rng(7)
    x, wt, b = values(rng, (1, 12, 13, 16), dt), values(rng, (20, 3, 3, 16), dt, 0.1), values(rng, (20,), dt)
    special = np.array([0x7f80, 0x7fc0], np.uint16) if dt == abi.BF16 else np.array([np.inf, np.nan], x.dtype)
    x[0, 0, 5, 3], x[0, 7, 12, 9] = special
    attr = abi.conv2d_attr((1, 1, 1, 1), acc_type=abi.ACC_F32)
    got = floats(run.conv2d(x, wt, b, (1, 12, 13, 20), dt, attr))
    want = floats(oracle.conv2d(x, wt, b, (1, 12, 13, 20), dt, attr))
    np.testing.assert_allclose(got, want, rtol=1.01 * STEP[dt], atol=2e-5)
    assert np.isnan(want).sum() == 20 * 6 and np.isinf(want).sum() == 20 * 6
