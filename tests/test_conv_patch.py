"""CONV2D (+RESCALE +CLAMP), CONCAT in front of it and TRANSPOSE_CONV2D with kernel = stride from a piece of the image in
shared memory: tile and patch edges, channel counts in every chunk width, several taps per piece, several channel blocks."""
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


CONV = [
    # n, h, w, ic, oc, kernel, stride, dilation, pad
    (1, 9, 33, 3, 24, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),      # four bytes a pixel, three taps a piece
    (2, 8, 17, 4, 33, (5, 5), (2, 2), (1, 1), (2, 2, 2, 2)),      # two pieces a kernel row
    (1, 11, 21, 7, 9, (3, 5), (1, 2), (2, 1), (2, 2, 2, 2)),      # eight bytes a pixel
    (1, 16, 16, 8, 64, (2, 2), (1, 1), (1, 1), (0, 1, 0, 1)),
    (1, 7, 64, 5, 3, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0)),
    (3, 13, 9, 20, 20, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),     # dwords, an odd number of pieces
    (1, 10, 40, 24, 70, (3, 3), (2, 2), (1, 1), (0, 1, 0, 1)),    # eight-byte chunks, three channel blocks, ragged
    (1, 12, 31, 48, 96, (3, 3), (1, 1), (2, 2), (2, 2, 2, 2)),    # 16-byte chunks, whole channel blocks
    (2, 6, 70, 33, 21, (1, 3), (1, 1), (1, 1), (0, 0, 1, 1)),
    (1, 5, 130, 29, 17, (7, 1), (1, 1), (1, 1), (3, 3, 0, 0)),
    (1, 200, 180, 12, 40, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),  # blocks that walk several tiles
    (1, 1, 1, 16, 5, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),
]


@pytest.mark.parametrize("case", CONV, ids=["_".join(map(str, c[1:5] + c[5] + c[6])) for c in CONV])
def test_conv2d_from_image_pieces_vs_oracle(dev, oracle, case):
    n, h, w, ic, oc, (kh, kw), (sy, sx), (dy, dx), pad = case
    run, rng = Runner(dev), np.random.default_rng(zlib.crc32(repr(case).encode()))
    x, wt = i8(rng, (n, h, w, ic)), i8(rng, (oc, kh, kw, ic))
    b = rng.integers(-2 ** 12, 2 ** 12, (oc,)).astype(np.int32)
    shape = (n, (h + pad[0] + pad[1] - (kh - 1) * dy - 1) // sy + 1, (w + pad[2] + pad[3] - (kw - 1) * dx - 1) // sx + 1, oc)
    attr = abi.conv2d_attr(pad, (sy, sx), (dy, dx), -5, 0)
    mult, shift = scale(rng, oc, kh * kw * ic)
    rattr = abi.rescale_attr(0, 3, True, True, True)
    exp = np.clip(oracle.rescale(oracle.conv2d(x, wt, b, shape, abi.I32, attr), mult, shift, abi.I8, rattr), -100, 90)
    np.testing.assert_array_equal(run.conv2d(x, wt, b, shape, abi.I8, attr, epilogue=(mult, shift, rattr, (-100, 90))), exp)


@pytest.mark.parametrize("h, w, ic, c1, c2, oc, s", [(9, 20, 24, 24, 24, 24, (2, 2)), (5, 33, 13, 12, 20, 19, (2, 3)),
                                                      (16, 8, 48, 32, 16, 40, (3, 1)), (4, 5, 7, 36, 4, 80, (1, 2))])
def test_transposed_convolution_and_concat_from_image_pieces(dev, h, w, ic, c1, c2, oc, s):
    rng = np.random.default_rng(h * 100 + ic)
    spec = graphs.Spec()
    spec.inputs += [("low", abi.I8, (2, h, w, ic)), ("skip", abi.I8, (2, s[0] * h, s[1] * w, c2))]
    acc = spec.tensor("acc", abi.I32, (2, s[0] * h, s[1] * w, c1))
    spec.op("TRANSPOSE_CONV2D", ["low", spec.const("w", i8(rng, (c1,) + s + (ic,))), spec.const("b", np.arange(c1, dtype=np.int32))],
            [acc], [0, 0, 0, 0, s[0], s[1], -4, 0, abi.ACC_I32])
    up = fused.requant(spec, rng, acc, ic, clamp=(-90, 100))
    cat = spec.tensor("cat", abi.I8, (2, s[0] * h, s[1] * w, c1 + c2))
    spec.op("CONCAT", [up, "skip"], [cat], [3])
    acc = spec.tensor("acc", abi.I32, (2, s[0] * h, s[1] * w, oc))
    spec.op("CONV2D", [cat, spec.const("w", i8(rng, (oc, 3, 3, c1 + c2))), spec.const("b", np.arange(oc, dtype=np.int32))], [acc],
            [1, 1, 1, 1, 1, 1, 1, 1, 3, 0, abi.ACC_I32])
    fused.requant(spec, rng, acc, 9 * (c1 + c2), out="output")
    spec.outputs.append(("output", abi.I8, (2, s[0] * h, s[1] * w, oc)))
    names = fused.both_ways(dev, spec, {"low": i8(rng, (2, h, w, ic)), "skip": i8(rng, (2, s[0] * h, s[1] * w, c2))})
    assert names == ["TRANSPOSE_CONV2D+RESCALE+CLAMP", "CONCAT+CONV2D+RESCALE"]
