"""MAX_POOL2D and AVG_POOL2D over fp16, bf16 and fp32 images: windows of a few taps and global averages, padding, odd
sizes, NaN handling, against the oracle."""
import numpy as np
import pytest

from hip_util import Runner, abi, gpu_available, hb

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.fixture(scope="module")
def run():
    dev = hb.Device(0)
    yield Runner(dev)
    dev.close()


CASES = [  # type, image, kernel, stride, pad
    ("f16", (2, 12, 14, 16), (2, 2), (2, 2), (0, 0, 0, 0)),
    ("f16", (3, 7, 9, 8), (3, 3), (2, 1), (1, 1, 1, 1)),
    ("f16", (2, 14, 14, 72), (14, 14), (1, 1), (0, 0, 0, 0)),
    ("f16", (1, 8, 4, 24), (8, 4), (1, 1), (0, 0, 0, 0)),
    ("f16", (1, 33, 5, 8), (7, 5), (1, 1), (3, 3, 2, 2)),
    ("bf16", (2, 9, 10, 40), (3, 2), (3, 2), (0, 0, 0, 0)),
    ("bf16", (1, 7, 13, 16), (7, 13), (1, 1), (0, 0, 0, 0)),
    ("f32", (2, 6, 5, 4), (2, 3), (1, 1), (1, 0, 1, 1)),
    ("f32", (5, 7, 13, 96), (7, 13), (1, 1), (0, 0, 0, 0)),
    ("f32", (1, 3, 3, 5), (3, 3), (1, 1), (0, 0, 0, 0)),  # rows no thread reads whole
]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}_{'x'.join(map(str, c[1] + c[2]))}" for c in CASES])
def test_float_pools_equal_the_oracle(run, oracle, case):
    kind, shape, kernel, stride, pad = case
    rng = np.random.default_rng(sum(shape) + kernel[0])
    x = rng.standard_normal(shape).astype(np.float32)
    if kind == "bf16":
        x = abi.typed((x.view(np.uint32) >> 16).astype(np.uint16), abi.BF16)
    else:
        x = x.astype({"f16": np.float16, "f32": np.float32}[kind])
    oh = (shape[1] + pad[0] + pad[1] - kernel[0]) // stride[0] + 1
    ow = (shape[2] + pad[2] + pad[3] - kernel[1]) // stride[1] + 1
    out = (shape[0], oh, ow, shape[3])

    def f32(a):
        return (np.asarray(a).astype(np.uint32) << 16).view(np.float32) if kind == "bf16" else np.asarray(a, np.float32)

    attr = abi.pool2d_attr(kernel, stride, pad, acc_type=abi.ACC_F32)
    got, want = f32(run.pool("avg_pool2d", x, out, attr)), f32(oracle.avg_pool2d(x, out, attr))
    eps = {"f16": 2.0 ** -11, "bf16": 2.0 ** -7, "f32": 1e-6}[kind]  # one rounding of the result, bf16 truncates
    np.testing.assert_allclose(got, want, rtol=2 * eps, atol=eps / 4)
    for nan_mode in (abi.NAN_PROPAGATE, abi.NAN_IGNORE):
        y = x.copy()
        y[:, ::2, :1, ::3] = {"bf16": 0x7fc0}.get(kind, np.nan)
        attr = abi.pool2d_attr(kernel, stride, pad, nan_mode=nan_mode)
        got, want = f32(run.pool("max_pool2d", y, out, attr)), f32(oracle.max_pool2d(y, out, attr))
        np.testing.assert_array_equal(got, want)
