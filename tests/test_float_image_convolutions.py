"""Floating-point convolutions of a few channels whose operands come straight from memory (conv_runs_float_kernel): pieces that
reach in front of the image's first byte and beyond the last, every number of steps, one and two groups of channels to a
wavefront, one bias for all, infinities beside the border, CLAMP on the way out."""
import importlib
import zlib

import numpy as np
import pytest

import test_fused_image_graphs as fused
import test_nonfinite_weights as nonfinite
from hip_util import gpu_available
from test_float_contractions import STEP, TYPES, abi, floats, run, values  # noqa: F401

graphs = fused.graphs
hb = importlib.import_module("ai-ml-emulation-layer-for-vulkan_amd.hip_backend")
pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]
IDS = ["f16", "bf16", "f32"]

CASES = [
    # n, h, w, ic, oc, kernel, stride, dilation, pad: at least 704 sub-tiles of 32 x 32
    (1, 151, 160, 3, 24, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),
    (2, 149, 151, 3, 64, (3, 3), (2, 2), (1, 1), (1, 1, 1, 1)),   # two groups of channels, a wavefront each
    (1, 259, 257, 1, 72, (2, 3), (1, 1), (1, 1), (0, 1, 1, 1)),   # and one for both, the last of eight channels
    (1, 150, 170, 3, 16, (5, 5), (1, 1), (1, 1), (2, 2, 2, 2)),   # five steps (fp32: a piece too many, stays)
    (1, 153, 152, 5, 8, (3, 3), (1, 1), (2, 1), (2, 2, 1, 1)),    # dilated along the column; fp32: six steps
    (3, 101, 80, 2, 32, (4, 2), (1, 1), (1, 1), (0, 0, 0, 0)),    # no border
    (1, 40, 700, 3, 8, (3, 3), (1, 1), (1, 1), (4, 4, 5, 5)),     # positions that meet no pixel
    # more pieces: what stays without stages
    (1, 262, 260, 4, 16, (5, 5), (1, 1), (1, 1), (2, 2, 2, 2)),   # eight steps, more than 2048 sub-tiles of 32 channels at most
    (1, 258, 257, 7, 24, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),   # five, rows that are no whole words (fp32: a piece too many)
    (1, 90, 84, 6, 88, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),     # five of an even number of channels (fp32: eight, with stages)
    (1, 90, 84, 7, 88, (3, 3), (1, 1), (1, 1), (1, 1, 1, 1)),     # and of an odd one: with stages
    (1, 90, 84, 4, 88, (4, 4), (1, 1), (1, 1), (2, 1, 1, 2)),     # four: with stages
    (1, 92, 88, 2, 88, (7, 7), (1, 1), (1, 1), (0, 0, 0, 0)),     # no border: seven of an even number of channels, without
    (1, 130, 129, 7, 264, (5, 2), (1, 1), (1, 1), (0, 0, 0, 0)),  # five of an odd one, two pieces a row, two groups of channels
]


@pytest.mark.parametrize("one_bias", [False, True], ids=["", "one_bias"])
@pytest.mark.parametrize("dt", TYPES, ids=IDS)
@pytest.mark.parametrize("case", CASES, ids=["_".join(map(str, c[1:5] + c[5] + c[6])) for c in CASES])
def test_against_the_oracle(run, oracle, case, dt, one_bias):  # noqa: F811
    n, h, w, ic, oc, (kh, kw), (sy, sx), (dy, dx), pad = case
    rng = np.random.default_rng(zlib.crc32(repr(case).encode()) + dt)
    x, wt = values(rng, (n, h, w, ic), dt), values(rng, (oc, kh, kw, ic), dt, (kh * kw * ic) ** -0.5)
    b = values(rng, (1 if one_bias else oc,), dt)
    shape = (n, (h + pad[0] + pad[1] - (kh - 1) * dy - 1) // sy + 1, (w + pad[2] + pad[3] - (kw - 1) * dx - 1) // sx + 1, oc)
    attr = abi.conv2d_attr(pad, (sy, sx), (dy, dx), acc_type=abi.ACC_F32)
    got, exp = floats(run.conv2d(x, wt, b, shape, dt, attr)), floats(oracle.conv2d(x, wt, b, shape, dt, attr))
    assert np.all(np.abs(got - exp) <= 2e-5 + 1.01 * STEP[dt] * np.abs(exp)), np.abs(got - exp).max()


@pytest.mark.parametrize("dt", TYPES, ids=IDS)
@pytest.mark.parametrize("case", [CASES[0], CASES[2]], ids=["narrow", "wide"])
def test_weights_that_are_not_finite(run, oracle, case, dt):  # noqa: F811
    nonfinite.test_weights_that_are_not_finite(run, oracle, case, dt)


@pytest.mark.parametrize("dt", [abi.F16, abi.F32], ids=["f16", "f32"])
def test_clamp_on_the_way_out(dt):
    rng, shape = np.random.default_rng(5), (1, 152, 150, 24)
    spec = graphs.Spec()
    spec.inputs.append(("x", dt, (1, 152, 150, 3)))
    acc = spec.tensor("acc", dt, shape)
    spec.op("CONV2D", ["x", spec.const("w", values(rng, (24, 3, 3, 3), dt, 0.2)), spec.const("b", values(rng, (24,), dt))], [acc],
            [1, 1, 1, 1, 1, 1, 1, 1, 0, 0, abi.ACC_F32])
    spec.op("CLAMP", [acc], ["output"], [abi.NAN_PROPAGATE], [0.0, 0.75])
    spec.outputs.append(("output", dt, shape))
    x = values(rng, (1, 152, 150, 3), dt)
    x[0, 70, 80, 1], x[0, 151, 149, 2] = np.nan, np.inf
    dev = hb.Device(0)
    try:
        assert fused.both_ways(dev, spec, {"x": x}) == ["CONV2D+CLAMP"]
    finally:
        dev.close()
