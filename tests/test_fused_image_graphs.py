"""Fusions of image-to-image graphs: CONCAT + CONV2D, TRANSPOSE_CONV2D + RESCALE + CLAMP, RESIZE + RESCALE (+ ARGMAX) and
floating-point CONV2D + ADD + CLAMP give the bits of the operators run one after another."""
import importlib

import numpy as np
import pytest

from hip_util import Runner, gpu_available

abi = importlib.import_module("ai-ml-emulation-layer-for-vulkan_amd.abi")
hb = importlib.import_module("ai-ml-emulation-layer-for-vulkan_amd.hip_backend")
graphs = importlib.import_module("ai-ml-emulation-layer-for-vulkan_amd.graphs")

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.fixture(scope="module")
def dev():
    d = hb.Device(0)
    yield d
    d.close()


def both_ways(dev, spec, inputs):
    outs = []
    for fuse in (False, True):
        g = graphs.build(dev, spec, fuse=fuse)
        for name, value in inputs.items():
            g.set_input(name, value)
        g.dispatch()
        dev.sync()
        outs.append(({name: g.get_output(name) for name, _, _ in spec.outputs}, g.op_names()))
        g.close()
    (plain, _), (fused, names) = outs
    for name in plain:
        np.testing.assert_array_equal(fused[name], plain[name])
    return names


def requant(spec, rng, acc, taps, out=None, clamp=None):
    shape = spec.shape_of(acc)
    mult = spec.const("m", rng.integers(2 ** 30, 2 ** 31 - 1, (shape[3],)).astype(np.int32))
    shift = spec.const("s", np.full((shape[3],), 31 + int(np.log2(100 * taps ** 0.5)), np.int8))
    y = out if out and clamp is None else spec.tensor("r", abi.I8, shape)
    spec.op("RESCALE", [acc, mult, shift], [y], [0, 2, 1, 1, 1, 0, 0])
    if clamp is None:
        return y
    z = out or spec.tensor("y", abi.I8, shape)
    spec.op("CLAMP", [y], [z], [abi.NAN_PROPAGATE], list(clamp))
    return z


@pytest.mark.parametrize("c1, c2, oc, k", [(16, 16, 24, 3), (5, 13, 19, 3), (40, 3, 33, 1), (1, 64, 8, 3)])
def test_concat_and_transposed_convolution_in_one_launch(dev, c1, c2, oc, k):
    rng = np.random.default_rng(c1 * 100 + c2)
    n, h, w = 2, 6, 7
    spec = graphs.Spec()
    spec.inputs += [("low", abi.I8, (n, h, w, 9)), ("skip", abi.I8, (n, 2 * h, 2 * w, c2))]
    i8 = lambda shape: rng.integers(-127, 127, shape, endpoint=True).astype(np.int8)
    acc = spec.tensor("acc", abi.I32, (n, 2 * h, 2 * w, c1))
    spec.op("TRANSPOSE_CONV2D", ["low", spec.const("w", i8((c1, 2, 2, 9))), spec.const("b", np.arange(c1, dtype=np.int32))], [acc],
            [0, 0, 0, 0, 2, 2, -4, 0, abi.ACC_I32])
    up = requant(spec, rng, acc, 9, clamp=(-90, 100))
    cat = spec.tensor("cat", abi.I8, (n, 2 * h, 2 * w, c1 + c2))
    spec.op("CONCAT", [up, "skip"], [cat], [3])
    acc = spec.tensor("acc", abi.I32, (n, 2 * h, 2 * w, oc))
    p = k // 2
    spec.op("CONV2D", [cat, spec.const("w", i8((oc, k, k, c1 + c2))), spec.const("b", np.arange(oc, dtype=np.int32))], [acc],
            [p, p, p, p, 1, 1, 1, 1, 3, 0, abi.ACC_I32])
    requant(spec, rng, acc, k * k * (c1 + c2), out="output")
    spec.outputs.append(("output", abi.I8, (n, 2 * h, 2 * w, oc)))
    names = both_ways(dev, spec, {"low": i8((n, h, w, 9)), "skip": i8((n, 2 * h, 2 * w, c2))})
    assert names == ["TRANSPOSE_CONV2D+RESCALE+CLAMP", "CONCAT+CONV2D+RESCALE"]


@pytest.mark.parametrize("argmax", [False, True], ids=["image", "labels"])
@pytest.mark.parametrize("c, up, mult", [(1, 2, 2 ** 30), (19, 2, 2 ** 30), (6, 3, 1908874354), (8, 4, 2 ** 30), (21, 2, -2 ** 30)])
def test_resize_rescale_argmax_in_one_launch(dev, c, up, mult, argmax):
    rng = np.random.default_rng(c)
    n, h, w = 2, 7, 9
    spec = graphs.Spec()
    spec.inputs.append(("input", abi.I8, (n, h, w, c)))
    big = (n, up * h, up * w, c)
    wide = spec.tensor("wide", abi.I32, big)
    spec.op("RESIZE", ["input"], [wide], [2 * up, 2, 2 * up, 2, 1 - up, 1 - up, up - 1, up - 1, 2])
    score = spec.tensor("score", abi.I8, big) if argmax else "output"
    scale = [spec.const("m", np.array([mult], np.int32)), spec.const("s", np.array([36 if up == 3 else 34], np.int8))]
    spec.op("RESCALE", [wide] + scale, [score], [0, 0, 1, 1, 0, 0, 0])
    if argmax:
        spec.op("ARGMAX", [score], ["output"], [3, abi.NAN_PROPAGATE])
        spec.outputs.append(("output", abi.I32, big[:3]))
    else:
        spec.outputs.append(("output", abi.I8, big))
    names = both_ways(dev, spec, {"input": rng.integers(-128, 127, (n, h, w, c), endpoint=True).astype(np.int8)})
    assert names == ["RESIZE+RESCALE" + ("+ARGMAX" if argmax else "")]


@pytest.mark.parametrize("rows, cols", [(3, 1), (70, 5), (9, 33), (4, 600), (2, 5000)])
def test_argmax_over_rows_vs_oracle(dev, oracle, rows, cols):
    run, rng = Runner(dev), np.random.default_rng(cols)
    few = rng.integers(-3, 3, (rows, cols)).astype(np.int8)  # many equal maxima
    for x in (few, few.astype(np.float16), few.astype(np.float32), np.full((rows, cols), -np.inf, np.float16)):
        np.testing.assert_array_equal(run.argmax(x, 1), oracle.argmax(x, 1))
    x = few.astype(np.float32)
    x[0, cols // 2] = np.nan
    for mode in (abi.NAN_PROPAGATE, abi.NAN_IGNORE):
        np.testing.assert_array_equal(run.argmax(x, 1, mode), oracle.argmax(x, 1, mode))


@pytest.mark.parametrize("dt", [abi.F16, abi.F32], ids=["f16", "f32"])
@pytest.mark.parametrize("ic, oc", [(16, 24), (3, 7)])
def test_convolution_addition_clamp_in_one_launch(dev, dt, ic, oc):
    rng = np.random.default_rng(ic)
    npdt, shape = abi.NP_OF[dt], (2, 9, 8, oc)
    spec = graphs.Spec()
    spec.inputs += [("x", dt, (2, 9, 8, ic)), ("r", dt, shape)]
    values = lambda s: rng.standard_normal(s).astype(npdt)
    y, z = spec.tensor("t", dt, shape), spec.tensor("t", dt, shape)
    spec.op("CONV2D", ["x", spec.const("w", values((oc, 3, 3, ic))), spec.const("b", values(oc))], [y],
            [1, 1, 1, 1, 1, 1, 1, 1, 0, 0, abi.ACC_F32])
    spec.op("ADD", ["r", y], [z])
    spec.op("CLAMP", [z], ["output"], [abi.NAN_PROPAGATE], [-1.5, 2.25])
    spec.outputs.append(("output", dt, shape))
    assert both_ways(dev, spec, {"x": values((2, 9, 8, ic)), "r": values(shape)}) == ["CONV2D+ADD+CLAMP"]
