"""Forms of the contraction kernels that only certain extents, layouts or result types reach: the large tile of K-major
floating-point products, requantised TRANSPOSE_CONV2D of several phases, and the byte-wise fetch of the staged int8 kernel."""
import ctypes as C
import zlib

import numpy as np
import pytest

from hip_util import gpu_available
from test_float_contractions import TYPES, abi, floats, run, values  # noqa: F401
from test_ragged_contractions import TCONV, i8, scale

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

LARGE = [
    # batches, m, k, n: at least one tile of 128 x 128 per compute unit (256), ragged in rows, columns and K
    (1, 2050, 33, 2060), (1, 2177, 200, 1921), (9, 643, 64, 667), (1, 2176, 131, 2048),
]


@pytest.mark.parametrize("row", [False, True], ids=["plain", "row"])
@pytest.mark.parametrize("dt", TYPES, ids=["f16", "bf16", "f32"])
@pytest.mark.parametrize("case", LARGE, ids=["x".join(map(str, c)) for c in LARGE])
def test_large_k_major_products(run, case, dt, row):  # noqa: F811
    nb, m, k, n = case
    assert nb * -(-m // 128) * -(-n // 128) >= 256
    rng = np.random.default_rng(zlib.crc32(repr(case).encode()))
    a, b = values(rng, (nb, m, k), dt), values(rng, (nb, k, n), dt)
    bias = rng.standard_normal((1, 1, n)).astype(np.float32)
    want = np.matmul(floats(a).astype(np.float64), floats(b).astype(np.float64)) + (bias if row else 0)
    ta, tb, tr, to = run.put(a), run.put(b), run.put(bias), run.new(abi.F32, (nb, m, n))
    attr = abi.MatmulAttr(0, 0)
    if row:
        run.dev.op("matmul_add", to.ref, ta.ref, tb.ref, C.byref(attr), tr.ref)
    else:
        run.dev.op("matmul", to.ref, ta.ref, tb.ref, C.byref(attr))
    got = to.download()
    run.done()
    # fp32 sums of k exact products (fp32: rounded ones), each of a size around one
    np.testing.assert_allclose(got, want, rtol=0, atol=3e-6 * np.sqrt(k) * max(1.0, np.abs(want).max()))


@pytest.mark.parametrize("zw", [0, 4])
@pytest.mark.parametrize("case", TCONV, ids=[c[0] for c in TCONV])
def test_transpose_conv2d_rescaled_vs_oracle(run, oracle, case, zw):  # noqa: F811
    """The requantised form of every case, most of which have several phases and a kernel that is not the stride."""
    name, n, h, w, ic, oc, (kh, kw), (sy, sx), pad = case
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    x, wt = i8(rng, (n, h, w, ic)), i8(rng, (oc, kh, kw, ic))
    b = rng.integers(-2 ** 12, 2 ** 12, (oc,)).astype(np.int32)
    shape = (n, (h - 1) * sy + pad[0] + pad[1] + kh, (w - 1) * sx + pad[2] + pad[3] + kw, oc)
    attr = abi.tconv2d_attr(pad, (sy, sx), 6, zw)
    mult, shift = scale(rng, oc, ic)
    rattr = abi.rescale_attr(0, 3, True, True, True)
    exp = oracle.rescale(oracle.transpose_conv2d(x, wt, b, shape, abi.I32, attr), mult, shift, abi.I8, rattr)
    tx, tw, tb, to = run.put(x), run.put(wt), run.put(b), run.new(abi.I8, shape)
    e = run._epi(mult, shift, rattr, (-100, 90))
    assert run.dev.lib.mlel_hip_transpose_conv2d_rescale_clamp_in_kernel(to.ref, tx.ref, tw.ref, tb.ref, C.byref(attr)) == 1
    run.dev.op("transpose_conv2d_rescale_clamp", to.ref, tx.ref, tw.ref, tb.ref, C.byref(attr), C.byref(e))
    got = to.download()
    run.done()
    np.testing.assert_array_equal(got, np.clip(exp, -100, 90))


PITCHED = [
    # name, n, h, w, ic, bytes per pixel, oc, kernel, split: images whose pixels lie apart, which the kernels for ragged rows decline
    ("split_k", 1, 8, 8, 232, 240, 24, 3, True),
    ("few_channels", 2, 9, 10, 6, 8, 40, 3, False),
    ("odd_pitch", 1, 20, 21, 21, 27, 130, 3, False),
    ("tall_tile", 4, 90, 91, 5, 9, 33, 1, False),
]


@pytest.mark.parametrize("zw", [0, 1])
@pytest.mark.parametrize("case", PITCHED, ids=[c[0] for c in PITCHED])
def test_conv2d_i8_of_pixels_that_lie_apart_vs_oracle(run, oracle, case, zw):  # noqa: F811
    name, n, h, w, ic, pitch, oc, k, split = case
    rng = np.random.default_rng(zlib.crc32(name.encode()))
    x, wt = i8(rng, (n, h, w, ic)), i8(rng, (oc, k, k, ic))
    b = rng.integers(-2 ** 12, 2 ** 12, (oc,)).astype(np.int32)
    attr = abi.conv2d_attr((k // 2,) * 4, (1, 1), (1, 1), 9, zw)
    strides, shape = (h * w * pitch, w * pitch, pitch, 1), (n, h, w, oc)
    acc = oracle.conv2d(x, wt, b, shape, abi.I32, attr)
    np.testing.assert_array_equal(run.conv2d(x, wt, b, shape, abi.I32, attr, x_strides=strides), acc)
    mult, shift = scale(rng, oc, k * k * ic)
    rattr = abi.rescale_attr(0, -2, True, True, True)
    for dt, less in ((abi.I8, 0), (abi.I16, 7)):
        epi = (mult, (shift - less).astype(np.int8), rattr, None)
        out = run.conv2d(x, wt, b, shape, dt, attr, epilogue=epi, x_strides=strides)
        np.testing.assert_array_equal(out, oracle.rescale(acc, *epi[:2], dt, rattr))
    # the entry point that says what it used: the staged kernel's partial tiles where K is split
    tx, tw, tb, to = run.put(x, strides=strides), run.put(wt), run.put(b), run.new(abi.I8, shape)
    e = run._epi(mult, shift, rattr, None)
    run.dev.op("conv2d_rescale_clamp_static", to.ref, tx.ref, tw.ref, tb.ref, C.byref(attr), C.byref(e))
    got = to.download()
    assert run.dev.lib.mlel_hip_static_scratch_last_use(run.dev.ctx) == int(split)
    run.done()
    np.testing.assert_array_equal(got, oracle.rescale(acc, mult, shift, abi.I8, rattr))


@pytest.mark.parametrize("b_rows", [False, True], ids=["k_major", "row_wise"])
@pytest.mark.parametrize("case", [(1, 37, 2100, 29), (3, 40, 53, 31), (2, 130, 135, 450)], ids=lambda c: "x".join(map(str, c)))
def test_matmul_i8_to_int16_vs_oracle(run, oracle, case, b_rows):  # noqa: F811
    """RESCALE to int16, which the product of ragged rows has no form of."""
    nb, m, k, n = case
    rng = np.random.default_rng(k)
    a, b = i8(rng, (nb, m, k)), i8(rng, (nb, k, n))
    mult, shift = scale(rng, 1, k)
    shift = (shift - 7).astype(np.int8)
    rattr = abi.rescale_attr(0, 3, True, True, False)
    out = run.matmul(a, b, abi.I16, 5, -5, epilogue=(mult, shift, rattr, None), b_rows=b_rows)
    np.testing.assert_array_equal(out, oracle.rescale(oracle.matmul(a, b, abi.I32, 5, -5), mult, shift, abi.I16, rattr))
