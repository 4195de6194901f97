"""int8 convolutions whose blocks have one tile of the image each (conv_patch_direct_i8_kernel): channel counts in every chunk
width and with every tail, tiles of every number of wavefronts and channels, rows shorter than a wavefront, borders, both sides
of the choice between it and the kernel whose blocks walk tiles."""
import zlib

import numpy as np
import pytest

import test_conv_few_tiles as few
from hip_util import Runner, abi, gpu_available, hb
from test_ragged_contractions import i8, scale

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.fixture(scope="module")
def dev():
    d = hb.Device(0)
    yield d
    d.close()


CASES = [
    # n, h, w, ic, oc, kernel, stride, dilation, pad, zero point
    (1, 150, 160, 4, 5, (3, 3), (1, 1), (1, 1), (0, 0, 0, 0), -128),
    (1, 149, 163, 12, 33, (5, 3), (1, 1), (2, 1), (4, 4, 1, 1), 127),       # dilated, a channel beyond 32
    (2, 130, 122, 24, 19, (3, 3), (2, 2), (1, 1), (0, 1, 0, 1), -5),
    (1, 3000, 9, 20, 24, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 9),          # several rows of a patch to a wavefront
    (1, 5, 6000, 8, 17, (3, 2), (1, 3), (1, 1), (1, 1, 0, 1), 0),
    (1, 221, 219, 20, 40, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -128),      # blocks of 64 channels
    (1, 340, 360, 12, 24, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 3),         # 256 positions
    (1, 120, 161, 96, 70, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -9),        # eight wavefronts, three channel blocks
    (1, 1050, 1010, 4, 3, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 2),         # eight wavefronts, one step
    (1, 150, 152, 60, 64, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -128),      # dwords, more of them than one round fetches
    (2, 113, 110, 64, 40, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 7),
    (1, 90, 100, 20, 20, (7, 7), (1, 1), (1, 1), (3, 3, 3, 3), -5),
    (1, 282, 281, 4, 300, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 5),         # many channels: blocks that walk tiles
    (1, 900, 890, 24, 7, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -7),         # many tiles of many steps: the same
    # 64 channels instead of the staged kernel: a result of 1 .. 32 channels modulo 64, of no whole dwords, many tiles
    (1, 130, 132, 64, 20, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 0),
    (1, 101, 99, 64, 39, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), -128),
    (1, 364, 362, 64, 36, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 5),
    (1, 190, 93, 64, 27, (2, 2), (1, 1), (1, 1), (0, 1, 0, 1), -5),
    (1, 262, 258, 56, 64, (3, 3), (1, 1), (2, 2), (2, 2, 2, 2), -3),        # 64 channels to a block where blocks walk tiles, 32 here: the same
    (1, 64, 190, 84, 20, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 6),          # a wide low tile would be fetched in too many turns
    (4, 105, 3, 68, 398, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1), 127),        # most of a tile outside the image: staged
    (1, 69, 177, 124, 64, (1, 1), (1, 1), (1, 1), (0, 0, 0, 0), 1),         # one tap, two: staged
    (1, 139, 41, 84, 186, (2, 1), (1, 1), (1, 1), (0, 0, 0, 0), -5),
]


@pytest.mark.parametrize("case", CASES, ids=["_".join(map(str, c[:5] + c[5] + c[6])) for c in CASES])
def test_conv2d_of_a_tile_per_block_vs_oracle(dev, oracle, case):
    n, h, w, ic, oc, (kh, kw), (sy, sx), (dy, dx), pad, zx = case
    run, rng = Runner(dev), np.random.default_rng(zlib.crc32(repr(case).encode()))
    x, wt = i8(rng, (n, h, w, ic)), i8(rng, (oc, kh, kw, ic))
    b = rng.integers(-2 ** 12, 2 ** 12, (oc,)).astype(np.int32)
    shape = (n, (h + pad[0] + pad[1] - (kh - 1) * dy - 1) // sy + 1, (w + pad[2] + pad[3] - (kw - 1) * dx - 1) // sx + 1, oc)
    attr = abi.conv2d_attr(pad, (sy, sx), (dy, dx), zx, 0)
    mult, shift = scale(rng, oc, kh * kw * ic)
    rattr = abi.rescale_attr(0, 3, True, True, True)
    exp = np.clip(oracle.rescale(oracle.conv2d(x, wt, b, shape, abi.I32, attr), mult, shift, abi.I8, rattr), -100, 90)
    np.testing.assert_array_equal(run.conv2d(x, wt, b, shape, abi.I8, attr, epilogue=(mult, shift, rattr, (-100, 90))), exp)


@pytest.mark.parametrize("case", [CASES[k] for k in (0, 2, 5, 7, 14, 12)],
                         ids=["4_channels", "stride", "64_to_a_block", "eight_wavefronts", "whole_pieces", "blocks_that_walk"])
def test_every_rescale_of_a_tile_per_block(dev, oracle, case):
    few.every_rescale(dev, oracle, case)


@pytest.mark.parametrize("n, h, w, ic, c1, c2, oc, s", [(1, 75, 81, 20, 12, 20, 36, (2, 2)), (2, 70, 75, 48, 32, 16, 24, (2, 2)),
                                                        (1, 40, 130, 64, 40, 56, 48, (3, 2)), (1, 180, 160, 24, 24, 24, 24, (2, 2))])
def test_two_images_and_transposed_convolution_of_a_tile_per_block(dev, n, h, w, ic, c1, c2, oc, s):
    few.test_two_images_and_transposed_convolution_of_few_tiles(dev, n, h, w, ic, c1, c2, oc, s)
