"""RESIZE with offsets that place positions in front of the image, and with a RESCALE whose input zero point makes its results
wrap: the one-launch kernels, the operators one by one and the oracle."""
import ctypes as C

import numpy as np
import pytest

import test_fused_image_graphs as fused
from hip_util import Runner, abi, gpu_available, hb

graphs = fused.graphs


@pytest.fixture(scope="module")
def dev():
    d = hb.Device(0)
    yield d
    d.close()


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("offset", [(-4, -4), (-5, 0), (0, -5), (-13, 1), (-9, -22), (-801, -402)], ids=lambda o: "%d_%d" % o)
def test_offsets_in_front_of_the_image(dev, oracle, offset):
    """Scale 4 / 2, offsets from one pixel to hundreds in front of the image: the second corner of a cell two or more in front
    is the last row or column (the shader's minimum is unsigned), as the operators give it one by one."""
    rng = np.random.default_rng(-offset[0])
    n, h, w, c = 2, 200, 331, 7
    big = (n, 2 * h, 2 * w, c)
    iattr = [4, 2, 4, 2, *offset, 0, 0, 2]
    spec = graphs.Spec()
    spec.inputs.append(("input", abi.I8, (n, h, w, c)))
    wide, score = spec.tensor("wide", abi.I32, big), spec.tensor("score", abi.I8, big)
    spec.op("RESIZE", ["input"], [wide], iattr)
    mult, shift = np.array([1500000011], np.int32), np.array([34], np.int8)
    spec.op("RESCALE", [wide, spec.const("m", mult), spec.const("s", shift)], [score], [0, 3, 1, 1, 0, 0, 0])
    spec.op("ARGMAX", [score], ["output"], [3, abi.NAN_PROPAGATE])
    spec.outputs.append(("output", abi.I32, big[:3]))
    values = rng.integers(-128, 127, (n, h, w, c), endpoint=True).astype(np.int8)
    assert fused.both_ways(dev, spec, {"input": values}) == ["RESIZE+RESCALE+ARGMAX"]
    want = oracle.resize(values, big, abi.I32, abi.resize_attr(iattr[:4], offset, (0, 0), 2))
    want = oracle.argmax(oracle.rescale(want, mult, shift, abi.I8, abi.rescale_attr(0, 3, True, True, False)), 3)
    g = graphs.build(dev, spec)
    g.set_input("input", values)
    g.dispatch()
    dev.sync()
    np.testing.assert_array_equal(g.get_output("output"), want)
    g.close()


# coordinates of the shader are int16: offsets beyond them wrap, which only the general kernel computes
FAR = [(-32001, 0), (0, -40000), (-70000, -65540)]


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("offset", FAR, ids=lambda o: "%d_%d" % o)
def test_offsets_beyond_int16_coordinates(dev, oracle, offset):
    values = np.random.default_rng(1).integers(-128, 127, (1, 9, 11, 5), endpoint=True).astype(np.int8)
    for mode, dt in ((1, abi.I8), (2, abi.I32)):
        attr = abi.resize_attr((1, 1, 1, 1), offset, (0, 0), mode)
        np.testing.assert_array_equal(Runner(dev).resize(values, (1, 9, 11, 5), dt, attr), oracle.resize(values, (1, 9, 11, 5), dt, attr))


@pytest.mark.parametrize("offset, taken", [((-32000, -32000), 1)] + [(o, 0) for o in FAR], ids=str)
def test_offsets_the_one_launch_form_takes(offset, taken):
    view = lambda dt, shape: abi.make_tensor(0, dt, shape)
    image, labels = view(abi.I8, (1, 9, 11, 5)), view(abi.I32, (1, 9, 11))
    attr = abi.resize_attr((1, 1, 1, 1), offset, (0, 0), 2)
    assert hb.load_library().mlel_hip_resize_rescale_in_kernel(C.byref(labels), C.byref(image), C.byref(attr), 1) == taken


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("zero_point", [0, 2 ** 21, -2 ** 21, 2 ** 31 - 1])
@pytest.mark.parametrize("h", [6, 400], ids=["few_labels", "many_labels"])
def test_labels_of_a_rescale_with_an_input_zero_point(dev, h, zero_point):
    """(a - 2^21) 2^10 leaves int32 on one side of zero: negative sums then scale to the largest value."""
    spec, big = graphs.Spec(), (1, 2 * h, 2 * 200, 7)
    spec.inputs.append(("input", abi.I8, (1, h, 200, 7)))
    wide, score = spec.tensor("wide", abi.I32, big), spec.tensor("score", abi.I8, big)
    spec.op("RESIZE", ["input"], [wide], [4, 2, 4, 2, -1, -1, 1, 1, 2])
    scale = [spec.const("m", np.array([2 ** 30], np.int32)), spec.const("s", np.array([20], np.int8))]
    spec.op("RESCALE", [wide] + scale, [score], [zero_point, 0, 1, 0, 0, 0, 0])
    spec.op("ARGMAX", [score], ["output"], [3, abi.NAN_PROPAGATE])
    spec.outputs.append(("output", abi.I32, big[:3]))
    values = np.random.default_rng(3).integers(-128, 127, (1, h, 200, 7), endpoint=True).astype(np.int8)
    assert fused.both_ways(dev, spec, {"input": values}) == ["RESIZE+RESCALE+ARGMAX"]


@pytest.mark.parametrize("w, c, taken", [(32767, 65536, 1), (32767, 65540, 0), (32000, 200000, 0)])
def test_rows_of_more_than_31_bits_are_left_to_the_general_kernel(w, c, taken):
    """A place within a row is an int32 in the one-launch kernels (judged without memory)."""
    image, out = (abi.make_tensor(0, abi.I8, shape) for shape in ((1, 2, w, c), (1, 2, 40, c)))
    attr = abi.resize_attr((1, 1, 1, 800), (0, 0), (0, 0), 2)
    assert hb.load_library().mlel_hip_resize_rescale_in_kernel(C.byref(out), C.byref(image), C.byref(attr), 0) == taken
