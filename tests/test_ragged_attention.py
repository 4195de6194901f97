"""mlel_hip_attention_rows_f16: numbers of queries and keys that are a multiple of nothing, against a float64 evaluation of
the chain's formula and, where the three launches take the case, bit for bit; the fusion of an encoder block of such a
length."""
import ctypes as C

import numpy as np
import pytest

import test_graph_host
from hip_util import Runner, abi, gpu_available, hb

graphs = test_graph_host.graphs


def _steps(scaled):
    o, f16 = (2 if scaled else 0), abi.F16
    steps = [(4, abi.RED["MAX"], o, 0, f16), (0, abi.BIN["SUB"], o, o + 1, f16), (2, abi.UN["EXP"], o + 2, 0, f16),
             (4, abi.RED["SUM"], o + 3, 0, f16), (2, abi.UN["RECIPROCAL"], o + 4, 0, f16), (1, 0, o + 3, o + 5, f16)]
    return ([(1, 0, 0, 1, f16)] if scaled else []) + steps


def _attention_rows(run, q, k, v, scale, merge):
    tq, tk, tv = run.put(q), run.put(k), run.put(v)
    c = abi.Chain()
    steps = _steps(scale is not None)
    c.n_inputs, c.n_steps = (1 if scale is None else 2), len(steps)
    if scale is not None:
        ts = run.put(np.array(scale, np.float16).reshape(1, 1, 1))
        c.inputs[1] = C.pointer(ts.view)
    for i, st in enumerate(steps):
        c.steps[i] = abi.ChainStep(*[int(x) for x in st])
    nb, m, _ = q.shape
    if not merge:
        to = run.new(abi.F16, (nb, m, 64))
        run.dev.op("attention_rows_f16", to.ref, tq.ref, tk.ref, tv.ref, C.byref(c))
    else:  # [1, nb, m, 64] -> [1, m, nb, 64]
        to = run.new(abi.F16, (m, nb, 64))
        view = abi.make_tensor(to.view.ptr, abi.F16, (1, nb, m, 1, 1, 64), (2 * m * nb * 64, 128, 2 * nb * 64, 0, 0, 2))
        run.dev.op("attention_rows_f16", C.byref(view), tq.ref, tk.ref, tv.ref, C.byref(c))
    r = to.download()
    run.done()
    return r.transpose(1, 0, 2) if merge else r


@pytest.fixture(scope="module")
def run():
    dev = hb.Device(0)
    yield Runner(dev)
    dev.close()


CASES = [(1, 1, 1), (3, 16, 17), (2, 63, 65), (3, 197, 197), (2, 65, 256), (2, 100, 257), (1, 64, 511), (2, 33, 513), (1, 130, 767),
         (1, 70, 1024)]


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="needs a GPU")
@pytest.mark.parametrize("merge", [False, True])
@pytest.mark.parametrize("case", CASES, ids=["h%d_m%d_s%d" % c for c in CASES])
@pytest.mark.parametrize("scale", [None, 0.125])
def test_any_number_of_queries_and_keys(run, case, scale, merge):
    nb, m, s = case
    rng = np.random.default_rng(nb * 1000003 + m * 1009 + s)
    q, k, v = (rng.standard_normal((nb, n, 64)).astype(np.float16) * np.float16(0.5) for n in (m, s, s))
    got = _attention_rows(run, q, k, v, scale, merge)
    x = (q.astype(np.float64) @ k.astype(np.float64).transpose(0, 2, 1)) * (1.0 if scale is None else scale)
    p = np.exp(x - x.max(-1, keepdims=True))
    want = (p / p.sum(-1, keepdims=True)) @ v.astype(np.float64)
    err = np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want)
    assert err < 4e-2, err  # every step of the chain rounds to fp16; the row sums add up in fp16
    if s % 8 == 0:
        chain_in = [run.matmul_bias_cast(q, np.ascontiguousarray(k.transpose(0, 2, 1)), None)]
        extra = [] if scale is None else [np.array(scale, np.float16).reshape(1, 1, 1)]
        prob = run.chain(chain_in + extra, _steps(scale is not None), chain_in[0].shape, abi.F16)
        np.testing.assert_array_equal(got.view(np.uint16), run.matmul_bias_cast(prob, v, None).view(np.uint16))


def test_encoder_blocks_of_any_length_fuse():
    """197 tokens: seven launches as at 512, K stored by rows; a graph that also reads the transposed keys keeps them."""
    three = " | ".join(["MATMUL+ADD+CAST+RESHAPE+TRANSPOSE"] * 3)
    attention = "MATMUL+CAST+ELEMENTWISE+REDUCE x7+MATMUL+CAST+RESHAPE+TRANSPOSE"
    g = test_graph_host._build_host_only(graphs.transformer_block_spec(batch=1, seq=197, d_model=384, heads=6, ffn=1536), fuse=True)
    assert g.op_names() == ["ELEMENTWISE+REDUCE x11", three, attention, "MATMUL+ADD+CAST+ADD", "ELEMENTWISE+REDUCE x11",
                            "MATMUL+ADD+CAST+ELEMENTWISE x9", "MATMUL+ADD+CAST+ADD"]
    g.close()
    spec = graphs.transformer_block_spec(batch=1, seq=197, d_model=128, heads=2, ffn=256)
    kt = next(op for op in spec.ops if op["op"] == "MATMUL" and spec.shape_of(op["out"][0]) == (2, 197, 197))["in"][1]
    spec.op("CAST", [kt], ["keys"])
    spec.outputs.append(("keys", abi.F32, (2, 64, 197)))
    g = test_graph_host._build_host_only(spec, fuse=True)
    assert attention not in g.op_names()
    g.close()
