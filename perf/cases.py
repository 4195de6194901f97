"""The work whose speed counts: data graphs and operators as a program on this framework runs them.

Every case goes through the public entry points (a GraphPipeline built with `graphs.build` and dispatched by a session,
or one operator of the C ABI through `hip_backend.Device.op`), with its inputs and its outputs in device memory and
everything a program keeps -- pipeline, session memory, constants -- made by `prepare`.  `listed` holds one fixed set;
`draw` gives more of the same ranges.
"""
import ctypes as C
import importlib
import math

import numpy as np
import torch

_PKG = "ai-ml-emulation-layer-for-vulkan_amd"
abi = importlib.import_module(_PKG + ".abi")
graphs = importlib.import_module(_PKG + ".graphs")

_DTYPES = {"i8": abi.I8, "f16": abi.F16, "bf16": abi.BF16, "f32": abi.F32}
_TORCH = {abi.I8: torch.int8, abi.I32: torch.int32, abi.F16: torch.float16, abi.BF16: torch.bfloat16,
          abi.F32: torch.float32}
_BYTES = {"i8": 1, "f16": 2, "bf16": 2, "f32": 4}

# multiply-adds of the largest case a draw may give: an int8 product of 4096^3, the encoder block of the benchmark, and
# 2048^3 for a floating-point product
_MOST_I8, _MOST_ENCODER, _MOST_FLOAT = 4096 ** 3, 32.3e9, 2048 ** 3


def listed():
    return [
        # One image at a time through the int8 classification network of the benchmark: latency, a chain of short
        # launches, recorded once and replayed as a serving loop does.
        {"name": "mobilenetv2_b1", "kind": "mobilenetv2", "batch": 1, "image": 224, "classes": 1000, "replayed": True},
        # The benchmark's batch, dispatched operator by operator.
        {"name": "mobilenetv2_b32", "kind": "mobilenetv2", "batch": 32, "image": 224, "classes": 1000, "replayed": False},
        # The fp16 encoder block of the benchmark: a large prefill.
        {"name": "encoder_b8_s512", "kind": "encoder", "batch": 8, "seq": 512, "heads": 12, "replayed": False},
        # A smaller encoder on one sequence of a length that is a multiple of nothing (image patches and a class token).
        {"name": "encoder_b1_s197", "kind": "encoder", "batch": 1, "seq": 197, "heads": 6, "replayed": True},
        # The benchmark's headline operator: batched int8 MATMUL with its RESCALE.
        {"name": "matmul_i8_b8_512x1024x1024", "kind": "matmul", "dtype": "i8", "batch": 8, "m": 512, "k": 1024, "n": 1024},
        # The same operator on a product that fills the device for many rounds.
        {"name": "matmul_i8_4096", "kind": "matmul", "dtype": "i8", "batch": 1, "m": 4096, "k": 4096, "n": 4096},
        # A bf16 projection over a ragged number of rows (fp32 result), as bf16 models run it.
        {"name": "matmul_bf16_b1_333x768x1001", "kind": "matmul", "dtype": "bf16", "batch": 1, "m": 333, "k": 768, "n": 1001},
        # One 3x3 int8 convolution with its per-channel RESCALE: the smallest call of the benchmark.
        {"name": "conv_i8_1x56x56x64", "kind": "conv", "batch": 1, "h": 56, "w": 56, "ic": 64, "oc": 64, "k": 3, "stride": 1},
        # Floating-point convolutions with residual additions, pooling and a classifier: a network before quantisation,
        # in half precision at a small batch ...
        {"name": "residual_f16_b4", "kind": "residual", "dtype": "f16", "batch": 4, "h": 224, "w": 224, "c": 64,
         "classes": 1000, "replayed": False},
        # ... and in single precision on one smaller image.
        {"name": "residual_f32_b1", "kind": "residual", "dtype": "f32", "batch": 1, "h": 112, "w": 208, "c": 24,
         "classes": 101, "replayed": False},
        # int8 image-to-image work, the everyday use of data graphs beside a renderer: strided convolutions down,
        # TRANSPOSE_CONV2D up with skip connections, RESIZE and ARGMAX behind it.  A thumbnail ...
        {"name": "segment_i8_64", "kind": "segment", "batch": 1, "h": 64, "w": 64, "c": 16, "classes": 21, "up": 2,
         "replayed": True},
        # ... and a frame.
        {"name": "segment_i8_360x640", "kind": "segment", "batch": 1, "h": 360, "w": 640, "c": 24, "classes": 19, "up": 2,
         "replayed": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mobilenetv2", "encoder", "matmul", "matmul", "conv", "residual", "segment"])
    while True:
        if kind == "mobilenetv2":
            return {"kind": kind, "batch": _log(rng, 1, 32), "image": 32 * rng.randint(3, 7), "classes": _log(rng, 10, 1001),
                    "replayed": rng.random() < 0.5}
        if kind == "encoder":
            c = {"kind": kind, "batch": _log(rng, 1, 8), "seq": _log(rng, 16, 768), "heads": rng.randint(3, 16),
                 "replayed": rng.random() < 0.5}
            if _encoder_macs(c) <= _MOST_ENCODER:
                return c
        if kind == "matmul":
            c = {"kind": kind, "dtype": rng.choice(["i8", "i8", "f16", "bf16", "f32"]), "batch": _log(rng, 1, 16),
                 "m": _log(rng, 1, 4096), "k": _log(rng, 16, 4096), "n": _log(rng, 16, 4096)}
            if c["batch"] * c["m"] * c["k"] * c["n"] <= (_MOST_I8 if c["dtype"] == "i8" else _MOST_FLOAT):
                return c
        if kind == "conv":
            c = {"kind": kind, "batch": _log(rng, 1, 16), "h": _log(rng, 7, 160), "w": _log(rng, 7, 160),
                 "ic": _log(rng, 3, 320), "oc": _log(rng, 8, 512), "k": rng.choice([1, 3, 3, 5]), "stride": 1}
            if c["h"] % 2 == 0 and c["w"] % 2 == 0:
                c["stride"] = rng.choice([1, 2])
            if c["batch"] * c["h"] * c["w"] * c["ic"] * c["oc"] * c["k"] ** 2 <= 20e9:
                return c
        if kind == "residual":
            c = {"kind": kind, "dtype": rng.choice(["f16", "f16", "f32"]), "batch": _log(rng, 1, 6),
                 "h": 16 * rng.randint(4, 16), "w": 16 * rng.randint(4, 16), "c": 8 * rng.randint(2, 8),
                 "classes": _log(rng, 10, 1001), "replayed": rng.random() < 0.5}
            if c["batch"] * c["h"] * c["w"] * c["c"] ** 2 <= (4 if c["dtype"] == "f16" else 1) * 224 * 224 * 64 ** 2:
                return c
        if kind == "segment":
            c = {"kind": kind, "batch": _log(rng, 1, 4), "h": 4 * _log(rng, 10, 128), "w": 4 * _log(rng, 10, 160),
                 "c": 4 * rng.randint(2, 8), "classes": _log(rng, 2, 40), "up": rng.choice([2, 3, 4]),
                 "replayed": rng.random() < 0.5}
            if c["batch"] * c["h"] * c["w"] * c["c"] ** 2 <= 360 * 640 * 24 ** 2:
                return c


# ---- the graphs ---------------------------------------------------------------------------------------------------


def _conv(spec, x, dtype, out_dtype, weights, bias, pad, stride, zp=0, transposed=False, out_hw=None):
    """CONV2D (or TRANSPOSE_CONV2D) of `x`; the result's extents follow from the attributes unless given."""
    n, h, w, _ = spec.shape_of(x)
    oc, k = weights.shape[0], weights.shape[1]
    oh, ow = out_hw or ((h + pad[0] + pad[1] - k) // stride + 1, (w + pad[2] + pad[3] - k) // stride + 1)
    y = spec.tensor("t", out_dtype, (n, oh, ow, oc))
    acc = abi.ACC_I32 if dtype == abi.I8 else abi.ACC_F32
    spec.op("TRANSPOSE_CONV2D" if transposed else "CONV2D", [x, spec.const("w", weights), spec.const("b", bias)], [y],
            list(pad) + [stride, stride] + ([] if transposed else [1, 1]) + [zp, 0, acc])
    spec.macs["dense"] += weights.size * n * (h * w if transposed else oh * ow)
    return y


def _same_pad(k, stride):
    return (k // 2, k // 2, k // 2, k // 2) if stride == 1 else (0, k - 2, 0, k - 2)


def _segment_spec(case, rng):
    """int8: two levels down and up with skip connections, a classifier per pixel, bilinear RESIZE and ARGMAX."""
    n, h, w, c, classes, up = (case[k] for k in ("batch", "h", "w", "c", "classes", "up"))
    spec = graphs.Spec()
    spec.inputs.append(("input", abi.I8, (n, h, w, 3)))

    def weights(oc, k, ic):
        return rng.integers(-127, 127, (oc, k, k, ic), endpoint=True).astype(np.int8)

    def requant(acc, taps, zp, relu):
        shape = spec.shape_of(acc)
        mult = rng.integers(2 ** 30, 2 ** 31 - 1, (shape[3],), endpoint=True).astype(np.int32)
        shift = np.full((shape[3],), 31 + int(round(math.log2(73 * math.sqrt(taps)))), np.int8)
        r = spec.tensor("r", abi.I8, shape)
        spec.op("RESCALE", [acc, spec.const("m", mult), spec.const("s", shift)], [r], [0, zp, 1, 1, 1, 0, 0])
        if not relu:
            return r
        y = spec.tensor("y", abi.I8, shape)
        spec.op("CLAMP", [r], [y], [abi.NAN_PROPAGATE], [zp, 127])
        return y

    def bias(oc):
        return rng.integers(-2 ** 12, 2 ** 12, (oc,), endpoint=True).astype(np.int32)

    def conv(x, zp, oc, k, stride=1, relu=True):
        ic = spec.shape_of(x)[3]
        acc = _conv(spec, x, abi.I8, abi.I32, weights(oc, k, ic), bias(oc), _same_pad(k, stride) if k > 1 else (0,) * 4,
                    stride, zp)
        return requant(acc, k * k * ic, -64, relu)

    def up2(x, skip, oc):
        _, xh, xw, ic = spec.shape_of(x)
        acc = _conv(spec, x, abi.I8, abi.I32, weights(oc, 2, ic), bias(oc), (0,) * 4, 2, -64, True, (2 * xh, 2 * xw))
        y = requant(acc, ic, -64, True)
        both = spec.tensor("cat", abi.I8, (n, 2 * xh, 2 * xw, oc + spec.shape_of(skip)[3]))
        spec.op("CONCAT", [y, skip], [both], [3])
        return both

    c0 = conv("input", -5, c, 3)
    c1 = conv(c0, -64, 2 * c, 3, 2)
    x = conv(conv(c1, -64, 4 * c, 3, 2), -64, 4 * c, 3)
    x = conv(up2(x, c1, 2 * c), -64, 2 * c, 3)
    x = conv(up2(x, c0, c), -64, c, 3)
    x = conv(x, -64, classes, 1, relu=False)
    wide = spec.tensor("wide", abi.I32, (n, up * h, up * w, classes))
    spec.op("RESIZE", [x], [wide], [2 * up, 2, 2 * up, 2, 1 - up, 1 - up, up - 1, up - 1, 2])
    score = spec.tensor("score", abi.I8, (n, up * h, up * w, classes))
    weight = 4 * up * up  # what the four corner weights of the RESIZE add up to
    s = 30 + math.ceil(math.log2(weight))
    scale = [spec.const("m", np.array([round(2 ** s / weight)], np.int32)), spec.const("s", np.array([s], np.int8))]
    spec.op("RESCALE", [wide] + scale, [score], [0, 0, 1, 1, 0, 0, 0])
    spec.op("ARGMAX", [score], ["output"], [3, abi.NAN_PROPAGATE])
    spec.outputs.append(("output", abi.I32, (n, up * h, up * w)))
    return spec


def _residual_spec(case, rng):
    """fp16 or fp32: stem, max pooling, residual blocks over three resolutions, global average, classifier."""
    dt, npdt = _DTYPES[case["dtype"]], abi.NP_OF[_DTYPES[case["dtype"]]]
    n, h, w, c, classes = (case[k] for k in ("batch", "h", "w", "c", "classes"))
    spec = graphs.Spec()
    spec.inputs.append(("input", dt, (n, h, w, 3)))

    def conv(x, oc, stride=1, gain=1.0):
        ic = spec.shape_of(x)[3]
        wt = (rng.standard_normal((oc, 3, 3, ic), dtype=np.float32) * (gain * math.sqrt(2.0 / (9 * ic)))).astype(npdt)
        return _conv(spec, x, dt, dt, wt, (0.1 * rng.standard_normal(oc)).astype(npdt), _same_pad(3, stride), stride)

    def relu(x):
        y = spec.tensor("y", dt, spec.shape_of(x))
        spec.op("CLAMP", [x], [y], [abi.NAN_PROPAGATE], [0.0, 6.0])
        return y

    def block(x):
        ch = spec.shape_of(x)[3]
        y = conv(relu(conv(x, ch)), ch, gain=0.5)
        z = spec.tensor("sum", dt, spec.shape_of(x))
        spec.op("ADD", [x, y], [z])
        return relu(z)

    x = relu(conv("input", c, 2))
    y = spec.tensor("pool", dt, (n, h // 4, w // 4, c))
    spec.op("MAX_POOL2D", [x], [y], [2, 2, 2, 2, 0, 0, 0, 0, abi.NAN_PROPAGATE])
    x = block(block(y))
    for ch in (2 * c, 4 * c):
        x = block(relu(conv(x, ch, 2)))
    _, ph, pw, ch = spec.shape_of(x)
    y = spec.tensor("mean", dt, (n, 1, 1, ch))
    spec.op("AVG_POOL2D", [x], [y], [ph, pw, 1, 1, 0, 0, 0, 0, abi.ACC_F32, 0, 0])
    flat = spec.tensor("flat", dt, (1, n, ch))
    spec.op("RESHAPE", [y], [flat])
    wt = spec.const("w", (rng.standard_normal((1, ch, classes), dtype=np.float32) / math.sqrt(ch)).astype(npdt))
    acc = spec.tensor("acc", abi.F32, (1, n, classes))
    spec.op("MATMUL", [flat, wt], [acc], [0, 0])
    spec.macs["dense"] += n * ch * classes
    spec.op("ADD", [acc, spec.const("b", (0.1 * rng.standard_normal((1, 1, classes))).astype(np.float32))], ["output"])
    spec.outputs.append(("output", abi.F32, (1, n, classes)))
    return spec


def _spec(case, seed):
    if case["kind"] == "mobilenetv2":
        return graphs.mobilenetv2_spec(case["batch"], case["image"], seed, True, case["classes"])
    if case["kind"] == "encoder":
        d = 64 * case["heads"]
        return graphs.transformer_block_spec(case["batch"], case["seq"], d, case["heads"], 4 * d, seed)
    return (_segment_spec if case["kind"] == "segment" else _residual_spec)(case, np.random.default_rng(seed))


def _encoder_macs(case):
    rows, d = case["batch"] * case["seq"], 64 * case["heads"]
    return rows * d * (12 * d + 2 * case["seq"])


# ---- what a program holds -----------------------------------------------------------------------------------------

_held = {}


def _device():
    """One context and one stream for the process, as a program has them."""
    if not _held:
        dev = importlib.import_module(_PKG + ".hip_backend").Device(0)
        _held["dev"], _held["stream"] = dev, dev.new_stream()
        dev.stream = _held["stream"]
    return _held["dev"]


class _Torch:
    """A torch tensor as an external tensor of a session and as an operand of an operator."""

    def __init__(self, t, dtype):
        self.t, self.ptr = t, t.data_ptr()
        self.view = abi.make_tensor(self.ptr, dtype, tuple(t.shape))
        self.ref = C.byref(self.view)


def _empty(dtype, shape):
    return _Torch(torch.empty(shape, dtype=_TORCH[dtype], device="cuda"), dtype)


def _random(gen, dtype, shape, lo=-128, hi=127):
    """Whole values over the type's range, or normal ones."""
    if dtype in (abi.I8, abi.I32):
        t = torch.randint(lo, hi + 1, shape, generator=gen, device="cuda", dtype=_TORCH[dtype])
    else:
        t = torch.randn(shape, generator=gen, device="cuda").to(_TORCH[dtype])
    return _Torch(t, dtype)


class _Graph:
    """A pipeline, one session of it and its bound tensors; `run` is one dispatch."""

    def __init__(self, case, seed, gen):
        dev = _device()
        spec = _spec(case, seed)
        self.g = graphs.build(dev, spec)
        self.s = self.g.new_session(allocate=False)
        self.s.bind_memory(self.g.session_mem)
        for name, dtype, shape in spec.inputs:
            self.s.bind(name, _random(gen, dtype, shape))
        for name, dtype, shape in spec.outputs:
            self.out = _empty(dtype, shape)
            self.s.bind(name, self.out)
        self.go = self.s.dispatch_replayed if case["replayed"] else self.s.dispatch

    def run(self):
        self.go()
        return self.out.t

    def __del__(self):
        self.s.close(free_tensors=False)
        self.g.close()


class _Op:
    """One operator of the C ABI on tensors that stay where they are; `run` is one call."""

    def __init__(self, case, seed, gen):
        self.dev = _device()
        rng = np.random.default_rng(seed)
        dtype = _DTYPES[case.get("dtype", "i8")]
        if case["kind"] == "conv":
            n, h, w, ic, oc, k, s = (case[x] for x in ("batch", "h", "w", "ic", "oc", "k", "stride"))
            pad = _same_pad(k, s) if k > 1 else (0, 0, 0, 0)
            x, wt = _random(gen, dtype, (n, h, w, ic)), _random(gen, dtype, (oc, k, k, ic), -127)
            bias = _random(gen, abi.I32, (oc,), -2 ** 15, 2 ** 15)
            self.out = _empty(dtype, (n,) + _conv_hw(case) + (oc,))
            attr, epi = abi.conv2d_attr(pad, (s, s), (1, 1), -5, 0), self._epilogue(rng, oc, k * k * ic, True)
            self.call = ("conv2d_rescale_clamp", self.out.ref, x.ref, wt.ref, bias.ref, C.byref(attr), C.byref(epi))
            self.keep = (x, wt, bias, attr, epi)
            return
        b, m, k, n = (case[x] for x in ("batch", "m", "k", "n"))
        x, y = _random(gen, dtype, (b, m, k)), _random(gen, dtype, (b, k, n))
        if dtype == abi.I8:
            self.out = _empty(dtype, (b, m, n))
            attr, epi = abi.MatmulAttr(2, -1), self._epilogue(rng, 1, k, False)
            self.call = ("matmul_rescale", self.out.ref, x.ref, y.ref, C.byref(attr), C.byref(epi))
        else:
            self.out = _empty(abi.F32, (b, m, n))
            attr, epi = abi.MatmulAttr(0, 0), None
            self.call = ("matmul", self.out.ref, x.ref, y.ref, C.byref(attr))
        self.keep = (x, y, attr, epi)

    def _epilogue(self, rng, channels, taps, per_channel):
        # a scale that leaves the results spread over int8
        mult = torch.from_numpy(rng.integers(2 ** 30, 2 ** 31 - 1, (channels,), endpoint=True).astype(np.int32)).cuda()
        shift = torch.full((channels,), 31 + int(round(math.log2(110 * math.sqrt(taps)))), dtype=torch.int8, device="cuda")
        self.scale = _Torch(mult, abi.I32), _Torch(shift, abi.I8)
        return self.dev.epilogue(self.scale[0], self.scale[1], abi.rescale_attr(0, 3, True, True, per_channel))

    def run(self):
        self.dev.op(*self.call)
        return self.out.t


def _conv_hw(case):
    k, s = case["k"], case["stride"]
    pad = _same_pad(k, s) if k > 1 else (0, 0, 0, 0)
    return (case["h"] + pad[0] + pad[1] - k) // s + 1, (case["w"] + pad[2] + pad[3] - k) // s + 1


# ---- the interface ------------------------------------------------------------------------------------------------


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return (_Op if case["kind"] in ("conv", "matmul") else _Graph)(case, seed, gen)


def run(state):
    return state.run()


def work(case):
    if case["kind"] == "matmul":
        b, m, k, n = (case[x] for x in ("batch", "m", "k", "n"))
        size = _BYTES[case["dtype"]]
        return {"bytes": b * (size * (m * k + k * n) + (1 if size == 1 else 4) * m * n), "flops": 2 * b * m * k * n}
    if case["kind"] == "conv":
        oh, ow = _conv_hw(case)
        n, h, w, ic, oc, k = (case[x] for x in ("batch", "h", "w", "ic", "oc", "k"))
        return {"bytes": n * h * w * ic + oc * k * k * ic + 9 * oc + n * oh * ow * oc,
                "flops": 2 * n * oh * ow * oc * k * k * ic}
    spec = _spec(case, 0)
    size = sum(a.nbytes for a in spec.consts.values())
    size += sum(abi.DTYPE_SIZE[dt] * math.prod(shape) for _, dt, shape in spec.inputs + spec.outputs)
    flops = spec.flops if case["kind"] == "encoder" else 2 * (spec.macs["dense"] + spec.macs["depthwise"])
    return {"bytes": size, "flops": flops}


def tolerance(case):
    if case["kind"] in ("mobilenetv2", "conv", "segment") or case.get("dtype") == "i8":
        return "exact"  # integer arithmetic
    if case["kind"] == "encoder" or (case["kind"] == "residual" and case["dtype"] == "f16"):
        return {"rel": 5e-3}  # every operator's result rounded to fp16
    return {"rel": 1e-5}  # fp32 sums of exact or fp32 products
