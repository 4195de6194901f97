"""The batch split over operators whose kernel reads at least 16 bytes of an image: halves of less are not split off."""
import numpy as np
import pytest

import test_fused_image_graphs as fused
import test_graph_host
from hip_util import abi, gpu_available, hb

graphs = fused.graphs


def spec_of(concat, ic):
    """TRANSPOSE_CONV2D + RESCALE, or CONCAT + CONV2D + RESCALE, of two images of 1 x 2 pixels of `ic` bytes, and a CLAMP."""
    rng = np.random.default_rng(ic)
    i8 = lambda shape: rng.integers(-127, 127, shape, endpoint=True).astype(np.int8)
    spec, image = graphs.Spec(), (2, 1, 2, ic)
    spec.inputs.append(("x", abi.I8, image))
    if concat:
        spec.inputs.append(("y", abi.I8, image))
        shape, both = (2, 1, 2, 5), spec.tensor("cat", abi.I8, (2, 1, 2, 2 * ic))
        spec.op("CONCAT", ["x", "y"], [both], [3])
        name, x, weights, iattr = "CONV2D", both, i8((5, 1, 1, 2 * ic)), [0, 0, 0, 0, 1, 1, 1, 1, 3, 0, abi.ACC_I32]
    else:
        shape = (2, 2, 4, 5)
        name, x, weights, iattr = "TRANSPOSE_CONV2D", "x", i8((5, 2, 2, ic)), [0, 0, 0, 0, 2, 2, -4, 0, abi.ACC_I32]
    acc = spec.tensor("acc", abi.I32, shape)
    spec.op(name, [x, spec.const("w", weights), spec.const("b", np.arange(5, dtype=np.int32))], [acc], iattr)
    y = fused.requant(spec, rng, acc, ic)
    spec.op("MAX_POOL2D", [y], ["output"], [1, 1, 1, 1, 0, 0, 0, 0, abi.NAN_PROPAGATE])
    spec.outputs.append(("output", abi.I8, shape))
    return spec, {n: i8(s) for n, _, s in spec.inputs}


@pytest.mark.parametrize("concat", [False, True], ids=["transposed", "concat"])
@pytest.mark.parametrize("ic, launches", [(7, 0), (8, 2)])
def test_what_is_split(concat, ic, launches):
    spec, _ = spec_of(concat, ic)
    g, _ = test_graph_host._build_split(spec)
    assert len(g.op_names()) == 2 and g.batch_split_launches() == launches
    g.close()


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("concat", [False, True], ids=["transposed", "concat"])
@pytest.mark.parametrize("ic", [7, 8])
def test_split_equals_the_whole(concat, ic):
    dev = hb.Device(0)
    spec, values = spec_of(concat, ic)
    outs = []
    for split in (False, True):
        g = graphs.build(dev, spec, split=split)
        for name, v in values.items():
            g.set_input(name, v)
        g.dispatch()
        dev.sync()
        outs.append(g.get_output("output"))
        g.close()
    np.testing.assert_array_equal(outs[1], outs[0])
    dev.close()
