"""int8 convolutions of few tiles (conv_few_i8_kernel): edges of tiles, stages and taps, every zero point's extremes, two images
side by side and TRANSPOSE_CONV2D, bit for bit against the oracle or the operators one by one."""
import zlib

import numpy as np
import pytest

import test_fused_image_graphs as fused
from hip_util import Runner, abi, gpu_available, hb
from test_ragged_contractions import i8, scale

graphs = fused.graphs
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.fixture(scope="module")
def dev():
    d = hb.Device(0)
    yield d
    d.close()


CASES = [
    # n, h, w, ic, oc, kernel, stride, dilation, pad, zero point, per channel
    (1, 1, 1, 16, 5, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -128, True),        # one position, one piece per tap
    (1, 5, 7, 16, 32, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 127, True),
    (2, 9, 6, 32, 17, (3, 3), (2, 2), (1, 1), (0, 1, 0, 1), 0, True),          # rows of 17 bytes
    (1, 8, 8, 48, 64, (5, 3), (1, 2), (2, 1), (4, 4, 1, 1), -5, False),        # three pieces per tap, dilated
    (3, 7, 7, 80, 30, (1, 1), (2, 2), (1, 1), (0, 0, 0, 0), 3, True),          # 1 x 1 with a stride
    (1, 14, 14, 128, 48, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -128, True),    # stages beyond the ring
    (1, 4, 4, 256, 132, (4, 4), (1, 1), (1, 1), (2, 1, 1, 2), 7, True),        # whole stages only
    (1, 60, 62, 32, 70, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -5, True),       # tiles of 32
    (2, 61, 50, 16, 33, (3, 3), (1, 1), (1, 1), (0, 2, 2, 0), -128, False),    # tiles of 32, ragged both ways
    (1, 30, 41, 144, 290, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 2, True),      # three tiles of 32 per unit
    (1, 90, 90, 64, 64, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -9, True),       # just beyond: the kernel of more tiles
    # channel counts that are no whole pieces: the ends of the operands, every remainder's masks, both depths of register sets
    (1, 3, 2, 3, 5, (2, 2), (1, 1), (1, 1), (0, 1, 1, 0), -128, True),
    (1, 4, 5, 17, 9, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 127, True),
    (2, 7, 6, 5, 33, (5, 5), (2, 1), (1, 1), (2, 2, 2, 2), -5, False),
    (1, 9, 9, 31, 32, (3, 3), (1, 1), (2, 2), (2, 2, 2, 2), 0, True),
    (3, 6, 7, 100, 40, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 9, True),
    (1, 12, 11, 44, 64, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), -128, True),
    (1, 50, 60, 37, 70, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -7, True),       # tiles of 32
    (1, 61, 63, 25, 100, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 4, False),      # tiles of 32, two per unit
    (4, 7, 35, 3, 144, (7, 7), (1, 1), (1, 1), (3, 3, 3, 3), -5, True),        # mostly padding: the kernel of image pieces
    (1, 9, 11, 3, 144, (7, 7), (1, 1), (1, 1), (3, 3, 3, 3), -5, True),        # the same, a tile of 16 per unit at most
]


@pytest.mark.parametrize("case", CASES, ids=["_".join(map(str, c[:5] + c[5] + c[6])) for c in CASES])
def test_conv2d_of_few_tiles_vs_oracle(dev, oracle, case):
    n, h, w, ic, oc, (kh, kw), (sy, sx), (dy, dx), pad, zx, per_channel = case
    run, rng = Runner(dev), np.random.default_rng(zlib.crc32(repr(case).encode()))
    x, wt = i8(rng, (n, h, w, ic)), i8(rng, (oc, kh, kw, ic))
    b = rng.integers(-2 ** 12, 2 ** 12, (oc if per_channel else 1,)).astype(np.int32)
    shape = (n, (h + pad[0] + pad[1] - (kh - 1) * dy - 1) // sy + 1, (w + pad[2] + pad[3] - (kw - 1) * dx - 1) // sx + 1, oc)
    attr = abi.conv2d_attr(pad, (sy, sx), (dy, dx), zx, 0)
    mult, shift = scale(rng, oc if per_channel else 1, kh * kw * ic)
    rattr = abi.rescale_attr(0, 3, True, True, per_channel)
    exp = np.clip(oracle.rescale(oracle.conv2d(x, wt, b, shape, abi.I32, attr), mult, shift, abi.I8, rattr), -100, 90)
    np.testing.assert_array_equal(run.conv2d(x, wt, b, shape, abi.I8, attr, epilogue=(mult, shift, rattr, (-100, 90))), exp)


def rescales(rng, oc, taps):
    """RESCALE as its multiplier, shift, attribute and CLAMP: 16-bit multipliers, one rounding, results without a sign."""
    for per_channel in (True, False):
        n = oc if per_channel else 1
        mult, shift = scale(rng, n, taps)
        mult16 = rng.integers(2 ** 14, 2 ** 15 - 1, (n,), endpoint=True).astype(np.int16)
        yield mult16, (shift - 16).astype(np.int8), abi.rescale_attr(0, -3, False, False, per_channel), (-100, 90)
        yield mult, shift, abi.rescale_attr(0, 3, True, False, per_channel), (-100, 90)
        yield mult, shift, abi.rescale_attr(0, 120, True, per_channel, per_channel, output_unsigned=True), None
        yield mult16, (shift - 16).astype(np.int8), abi.rescale_attr(0, 17, False, False, per_channel, output_unsigned=True), None


def every_rescale(dev, oracle, case):
    n, h, w, ic, oc, (kh, kw), (sy, sx), (dy, dx), pad, zx = case
    run, rng = Runner(dev), np.random.default_rng(zlib.crc32(repr(case).encode()))
    x, wt, b = i8(rng, (n, h, w, ic)), i8(rng, (oc, kh, kw, ic)), rng.integers(-2 ** 12, 2 ** 12, (oc,)).astype(np.int32)
    shape = (n, (h + pad[0] + pad[1] - (kh - 1) * dy - 1) // sy + 1, (w + pad[2] + pad[3] - (kw - 1) * dx - 1) // sx + 1, oc)
    attr = abi.conv2d_attr(pad, (sy, sx), (dy, dx), zx, 0)
    sums = oracle.conv2d(x, wt, b, shape, abi.I32, attr)
    for mult, shift, rattr, clamp in rescales(rng, oc, kh * kw * ic):
        exp = oracle.rescale(sums, mult, shift, abi.I8, rattr)
        if clamp is not None:
            exp = np.clip(exp, *clamp)
        got = run.conv2d(x, wt, b, shape, abi.I8, attr, epilogue=(mult, shift, rattr, clamp))
        np.testing.assert_array_equal(got.view(np.uint8), exp.astype(got.dtype, copy=False).view(np.uint8))
        assert len(np.unique(exp)) > 20


@pytest.mark.parametrize("case", [CASES[k][:-1] for k in (2, 5, 7, 15, 18)], ids=["rows_of_17", "three_stages", "tiles_of_32", "ragged", "ragged_tiles_of_32"])
def test_every_rescale_of_few_tiles(dev, oracle, case):
    every_rescale(dev, oracle, case)


@pytest.mark.parametrize("zx", [200, -129])
@pytest.mark.parametrize("ic", [64, 20], ids=["pieces", "ragged"])
def test_zero_points_that_are_no_byte(dev, oracle, ic, zx):
    """The zero point is subtracted in 32 bits, whatever its value: here as a factor of the weights' sums, without borders."""
    run, rng = Runner(dev), np.random.default_rng(ic)
    x, wt, b = i8(rng, (1, 9, 8, ic)), i8(rng, (24, 3, 3, ic)), rng.integers(-2 ** 12, 2 ** 12, (24,)).astype(np.int32)
    attr, rattr = abi.conv2d_attr((0, 0, 0, 0), (1, 1), (1, 1), zx, 0), abi.rescale_attr(0, 3, True, True, True)
    mult, shift = scale(rng, 24, 9 * ic)
    exp = np.clip(oracle.rescale(oracle.conv2d(x, wt, b, (1, 7, 6, 24), abi.I32, attr), mult, shift, abi.I8, rattr), -100, 90)
    np.testing.assert_array_equal(run.conv2d(x, wt, b, (1, 7, 6, 24), abi.I8, attr, epilogue=(mult, shift, rattr, (-100, 90))), exp)


@pytest.mark.parametrize("n, h, w, ic, c1, c2, oc, s", [
    (2, 3, 5, 16, 16, 16, 7, (1, 2)), (1, 6, 5, 16, 32, 16, 8, (3, 1)), (1, 8, 7, 64, 32, 48, 40, (2, 2)), (1, 4, 5, 32, 80, 16, 24, (3, 2)),
    (1, 40, 40, 48, 16, 16, 48, (2, 2)),      # tiles of 32
    (2, 5, 6, 13, 12, 20, 7, (2, 3)), (1, 7, 5, 24, 4, 36, 12, (1, 2)), (1, 30, 20, 28, 28, 28, 28, (2, 2)),  # no whole pieces
    (1, 120, 100, 48, 16, 32, 40, (2, 2)),    # more tiles than this kernel takes
])
def test_two_images_and_transposed_convolution_of_few_tiles(dev, n, h, w, ic, c1, c2, oc, s):
    rng = np.random.default_rng(h * 100 + ic)
    spec = graphs.Spec()
    spec.inputs += [("low", abi.I8, (n, h, w, ic)), ("skip", abi.I8, (n, s[0] * h, s[1] * w, c2))]
    acc = spec.tensor("acc", abi.I32, (n, s[0] * h, s[1] * w, c1))
    spec.op("TRANSPOSE_CONV2D", ["low", spec.const("w", i8(rng, (c1,) + s + (ic,))), spec.const("b", np.arange(c1, dtype=np.int32))],
            [acc], [0, 0, 0, 0, s[0], s[1], -4, 0, abi.ACC_I32])
    up = fused.requant(spec, rng, acc, ic, clamp=(-90, 100))
    cat = spec.tensor("cat", abi.I8, (n, s[0] * h, s[1] * w, c1 + c2))
    spec.op("CONCAT", [up, "skip"], [cat], [3])
    acc = spec.tensor("acc", abi.I32, (n, s[0] * h, s[1] * w, oc))
    spec.op("CONV2D", [cat, spec.const("w", i8(rng, (oc, 3, 3, c1 + c2))), spec.const("b", np.arange(oc, dtype=np.int32))], [acc],
            [1, 1, 1, 1, 1, 1, 1, 1, 3, 0, abi.ACC_I32])
    fused.requant(spec, rng, acc, 9 * (c1 + c2), out="output")
    spec.outputs.append(("output", abi.I8, (n, s[0] * h, s[1] * w, oc)))
    names = fused.both_ways(dev, spec, {"low": i8(rng, (n, h, w, ic)), "skip": i8(rng, (n, s[0] * h, s[1] * w, c2))})
    assert names == ["TRANSPOSE_CONV2D+RESCALE+CLAMP", "CONCAT+CONV2D+RESCALE"]
