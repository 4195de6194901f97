"""RESIZE + RESCALE + ARGMAX of an image large enough for the kernel that walks cells of four pixels: channel counts at the
edges of its fetches, fractional scales, equal maxima."""
import numpy as np
import pytest

import test_fused_image_graphs as fused
from hip_util import abi, gpu_available, hb

graphs = fused.graphs
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.fixture(scope="module")
def dev():
    d = hb.Device(0)
    yield d
    d.close()


@pytest.mark.parametrize("c, up, w", [(4, 2, 300), (19, 2, 257), (33, 3, 170), (50, 2, 260), (64, 4, 130)])
def test_resize_argmax_of_a_large_image(dev, c, up, w):
    rng = np.random.default_rng(c)
    n, h = 2, -(-2 ** 17 // (up * up * w)) + 1
    spec = graphs.Spec()
    spec.inputs.append(("input", abi.I8, (n, h, w, c)))
    big = (n, up * h, up * w, c)
    wide, score = spec.tensor("wide", abi.I32, big), spec.tensor("score", abi.I8, big)
    spec.op("RESIZE", ["input"], [wide], [2 * up, 2, 2 * up, 2, 1 - up, 1 - up, up - 1, up - 1, 2])
    # (clamped at both ends, and coarse: many equal maxima)
    scale = [spec.const("m", np.array([1500000011], np.int32)), spec.const("s", np.array([31 + (2 * up * up).bit_length()], np.int8))]
    spec.op("RESCALE", [wide] + scale, [score], [0, 3, 1, 1, 0, 0, 0])
    spec.op("ARGMAX", [score], ["output"], [3, abi.NAN_PROPAGATE])
    spec.outputs.append(("output", abi.I32, big[:3]))
    values = rng.integers(-128, 127, (n, h, w, c), endpoint=True).astype(np.int8)
    assert fused.both_ways(dev, spec, {"input": values}) == ["RESIZE+RESCALE+ARGMAX"]
