"""External tensors at addresses that are no multiple of 16: the fused operators whose kernels want aligned operands give the
bytes they give on aligned ones, dispatched and replayed, whole and with the batch split."""
import numpy as np
import pytest

import test_graph_host
from hip_util import abi, gpu_available, hb

graphs = test_graph_host.graphs


class Placed:
    """`array` (or zeros of `shape`) in device memory, `offset` bytes beyond an aligned address."""

    def __init__(self, dev, dtype, shape, offset, array=None):
        self.dev, self.shape, self.np = dev, shape, np.dtype(abi.NP_OF[dtype])
        self.bytes = int(np.prod(shape)) * self.np.itemsize
        self.base = dev.alloc(self.bytes + 64)
        self.ptr = self.base + offset
        guard = np.full(self.bytes + 64, 0x5a, np.uint8)
        if array is not None:
            guard[offset:offset + self.bytes] = np.ascontiguousarray(array).view(np.uint8).ravel()
        dev.h2d(self.base, guard.ctypes.data, guard.nbytes)
        self.offset = offset

    def download(self):
        raw = np.empty(self.bytes + 64, np.uint8)
        self.dev.d2h(raw.ctypes.data, self.base, raw.nbytes)
        assert (raw[:self.offset] == 0x5a).all() and (raw[self.offset + self.bytes:] == 0x5a).all()  # nothing around it written
        return raw[self.offset:self.offset + self.bytes].view(self.np).reshape(self.shape)

    def free(self):
        self.dev.free(self.base)


def attention_spec(heads, m, s, merge):
    """softmax(q k^T / 8) v with q, v and the result external; K arrives by rows and is transposed by the graph."""
    spec = graphs.Spec()
    f16, f32 = abi.F16, abi.F32
    spec.inputs += [("q", f16, (heads, m, 64)), ("k", f16, (heads, s, 64)), ("v", f16, (heads, s, 64))]

    def op(name, ins, dt, shape, iattr=()):
        y = spec.tensor("t", dt, shape)
        spec.op(name, ins, [y], list(iattr))
        return y

    kt = op("RESHAPE", [op("TRANSPOSE", ["k"], f16, (heads, 64, s), (0, 2, 1))], f16, (heads, 64, s))
    shape, row = (heads, m, s), (heads, m, 1)
    x = op("CAST", [op("MATMUL", ["q", kt], f32, shape, (0, 0))], f16, shape)
    x = op("MUL", [x, spec.const("c", np.full((1, 1, 1), 0.125, np.float16))], f16, shape, (0,))
    e = op("EXP", [op("SUB", [x, op("REDUCE_MAX", [x], f16, row, (2, abi.NAN_PROPAGATE))], f16, shape)], f16, shape)
    p = op("MUL", [e, op("RECIPROCAL", [op("REDUCE_SUM", [e], f16, row, (2,))], f16, row)], f16, shape, (0,))
    acc = op("MATMUL", [p, "v"], f32, (heads, m, 64), (0, 0))
    if merge:
        c = op("RESHAPE", [op("CAST", [acc], f16, (heads, m, 64))], f16, (1, heads, m, 64))
        spec.op("TRANSPOSE", [c], ["output"], [0, 2, 1, 3])
        spec.outputs.append(("output", f16, (1, m, heads, 64)))
    else:
        spec.op("CAST", [acc], ["output"])
        spec.outputs.append(("output", f16, (heads, m, 64)))
    return spec


def expansion_spec(n):
    """1x1 CONV2D + RESCALE and 3x3 DEPTHWISE_CONV2D + RESCALE, image and result external, and a pooling of the image (a batch
    is split from two launches on)."""
    rng = np.random.default_rng(n)
    h, w, ic, c = 9, 7, 32, 64
    spec = graphs.Spec()
    spec.inputs.append(("x", abi.I8, (n, h, w, ic)))
    i8 = lambda shape: rng.integers(-127, 127, shape, endpoint=True).astype(np.int8)

    def stage(op, x, weights, pad, taps, out):
        acc = spec.tensor("acc", abi.I32, (n, h, w, c))
        bias = spec.const("b", rng.integers(-2 ** 10, 2 ** 10, (c,)).astype(np.int32))
        spec.op(op, [x, spec.const("w", weights), bias], [acc], [pad] * 4 + [1, 1, 1, 1, 3, 0, abi.ACC_I32])
        mult = spec.const("m", rng.integers(2 ** 30, 2 ** 31 - 1, (c,)).astype(np.int32))
        shift = spec.const("s", np.full((c,), 31 + int(np.log2(100 * taps ** 0.5)), np.int8))
        spec.op("RESCALE", [acc, mult, shift], [out], [0, 2, 1, 1, 1, 0, 0])
        return out

    y = stage("CONV2D", "x", i8((c, 1, 1, ic)), 0, ic, spec.tensor("y", abi.I8, (n, h, w, c)))
    stage("DEPTHWISE_CONV2D", y, i8((3, 3, c, 1)), 1, 9, "output")
    spec.op("MAX_POOL2D", ["x"], ["pooled"], [3, 3, 1, 1, 1, 1, 1, 1, abi.NAN_PROPAGATE])
    spec.outputs += [("output", abi.I8, (n, h, w, c)), ("pooled", abi.I8, (n, h, w, ic))]
    return spec


ATTENTION = "MATMUL+CAST+ELEMENTWISE+REDUCE x7+MATMUL+CAST"
CASES = [
    # graph, operators after fusion, byte offset of the external tensors
    (lambda: attention_spec(3, 197, 197, False), ["TRANSPOSE", ATTENTION], 8),
    (lambda: attention_spec(2, 70, 130, True), ["TRANSPOSE", ATTENTION + "+RESHAPE+TRANSPOSE"], 2),
    (lambda: attention_spec(2, 64, 128, False), ["TRANSPOSE", ATTENTION], 8),
    (lambda: expansion_spec(2), ["CONV2D+RESCALE+DEPTHWISE_CONV2D+RESCALE", "MAX_POOL2D"], 3),
]
IDS = ["attention_ragged", "attention_merged", "attention_64", "expansion_depthwise"]


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("split", [False, True], ids=["whole", "split"])
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_external_tensors_at_any_address(case, split):
    make, names, offset = case
    dev = hb.Device(0)
    dev.stream = dev.new_stream()  # (a replayed dispatch is recorded on a stream of its own)
    spec, rng = make(), np.random.default_rng(5)
    g = graphs.build(dev, spec, split=split)
    assert g.op_names() == names and g.batch_split_launches() == (2 if split and "MAX_POOL2D" in names else 0)
    values = {name: rng.integers(-128, 127, shape).astype(np.int8) if dt == abi.I8 else rng.standard_normal(shape).astype(np.float16)
              for name, dt, shape in spec.inputs}
    results = []
    for off in (0, offset):
        s = g.new_session()
        held = {name: Placed(dev, dt, shape, off, values[name]) for name, dt, shape in spec.inputs}
        held.update({name: Placed(dev, dt, shape, off) for name, dt, shape in spec.outputs})
        for name, t in held.items():
            s.ext_tensors[name].free()
            s.bind(name, t)
        s.dispatch()
        dev.sync()
        results.append(held["output"].download())
        for _ in range(3):
            s.dispatch_replayed()
            dev.sync()
            np.testing.assert_array_equal(held["output"].download().view(np.uint8), results[-1].view(np.uint8))
        s.close()
    np.testing.assert_array_equal(results[1].view(np.uint8), results[0].view(np.uint8))
    assert np.unique(results[0].view(np.uint8)).size > 8
    g.close()
    dev.close()


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_stand_ins_live_for_one_launch(case):
    """Session memory for the external operands of such an operator and of no other, alive at that operator only."""
    make, names, _ = case
    spec = make()
    g = test_graph_host._build_host_only(spec, fuse=True)
    assert g.op_names() == names
    at = 1 + max(i for i, name in enumerate(names) if "+" in name)  # (position 0 belongs to the graph's inputs)
    extra = [t for t in g.session_tensors() if t["offset"] is not None and t["first"] == t["last"] == at]
    external = {"q", "v", "output"} if "q" in [i[0] for i in spec.inputs] else {"x", "output"}
    size = lambda dt, shape: int(np.prod(shape)) * abi.DTYPE_SIZE[dt]
    assert sorted(t["size"] for t in extra) == sorted(size(dt, sh) for n, dt, sh in spec.inputs + spec.outputs if n in external)
    g.close()
