"""The work this framework is used for, as cases that can be timed.

A case is one pass through a public entry point: the C ABI of libtbn_hip.so
(through the ctypes binding), the operator functions and the Session of the
_tbn module.  Kinds:

  linear  float x binary / float x ternary product on weights packed once
          (a fully connected layer: one row is one sample, thousands of rows a
          large batch), with the layer's scale, bias and ReLU
  dense   the fp32 GEMM of the layers that stay unquantized
  matmul  the operator qlinear_matmul_binary on a BINARY weight tensor, which
          packs the weights in every call
  tbn     the product in TBN arithmetic (activations ternarized at +-0.1,
          integer products), weights packed once
  conv    one convolution layer: binary or ternary weights in the conv layout
          (tile tuned once, as a Session does), fp32 weights, or TBN arithmetic
  model   a whole forward through a device-resident Session: LeNet (one 28x28
          image per sample) or ResNet-18 (224x224), returning the logits

Values follow the benchmark: activations N(0, 1), binary weights +-1 with
p = 0.5, ternary weights -1 / 0 / +1 with p = 0.3 / 0.4 / 0.3, scales
U[0.5, 1.5], biases N(0, 0.01).
"""
import ctypes
import pathlib
import sys

import numpy as np
import torch

_PKG = pathlib.Path(__file__).resolve().parents[1] / "fast-arm-tbcnn_amd"
for _p in (str(_PKG / "python"), str(_PKG / "lib")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import _tbn  # noqa: E402
import tbn_hip  # noqa: E402

DEVICE = "cuda:0"
TERNARIZE = 0.1  # TBN arithmetic: |v| above this keeps its sign


# ---- the cases ---------------------------------------------------------------------------


def _linear(name, weights, m, k, n, bias=False, relu=False):
    return {"name": name, "kind": "linear", "weights": weights, "m": m, "k": k, "n": n, "bias": bias, "relu": relu}


def _conv(name, weights, n, c, hw, m, k, stride=1, bias=True, relu=True, residual=False):
    return {"name": name, "kind": "conv", "weights": weights, "n": n, "c": c, "hw": hw, "m": m, "k": k,
            "stride": stride, "bias": bias, "relu": relu, "residual": residual}


def listed():
    return [
        # one digit through the smallest model: three kernels, all latency
        {"name": "lenet_1", "kind": "model", "model": "lenet", "batch": 1},
        # one sample through a large fully connected layer (online inference)
        _linear("linear_1", "binary", 1, 4096, 4096),
        # a hidden layer of odd sizes: rows that are not 16-byte aligned, no whole tiles
        _linear("linear_ragged", "binary", 777, 1333, 1001, bias=True, relu=True),
        # a ternary layer at a serving batch
        _linear("linear_ternary_256", "ternary", 256, 4096, 4096),
        # the headline product
        _linear("linear_4096", "binary", 4096, 4096, 4096),
        # a layer that stays fp32
        {"name": "dense_1024", "kind": "dense", "m": 1024, "k": 1024, "n": 1000, "bias": True, "trans_b": False},
        # the operator as the reference's users call it, BINARY weights packed per call
        {"name": "matmul_512", "kind": "matmul", "m": 512, "k": 2048, "n": 2048},
        # the reference's own arithmetic on the headline shape
        {"name": "tbn_4096", "kind": "tbn", "m": 4096, "k": 4096, "n": 4096},
        # the benchmark's conv layer
        _conv("conv_binary_14", "binary", 64, 64, 14, 128, 3),
        # a first-stage residual layer in TBN arithmetic
        _conv("conv_tbn_56", "tbn", 32, 64, 56, 64, 3, bias=False, residual=True),
        # the same kind of layer of a network run without quantization
        _conv("conv_f32_28", "f32", 16, 128, 28, 128, 3),
        # a whole network at the benchmark's batch
        {"name": "resnet18_32", "kind": "model", "model": "resnet18", "batch": 32},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choices(["linear", "dense", "matmul", "tbn", "conv", "model"], [30, 11, 10, 11, 30, 8])[0]
    if kind == "model":
        model = rng.choice(["lenet", "resnet18"])
        return {"kind": "model", "model": model, "batch": _log_int(rng, 1, 64 if model == "lenet" else 31)}
    if kind == "conv":
        weights = rng.choice(["binary", "ternary", "f32", "tbn"])
        c = _log_int(rng, 3 if weights == "f32" else 16, 512)
        hw = _log_int(rng, 7, 112)
        # the conv layout's patches: stride 2 up to 3x3 and from 33 output channels
        k = rng.choice([1, 3, 3, 5])
        stride = rng.choice([1, 1, 2]) if k < 5 else 1
        m = _log_int(rng, 16 if stride == 1 else 33, 512)
        n = _log_int(rng, 1, 64)
        out = (hw + 2 * (k // 2) - k) // stride + 1
        while n > 1 and 2.0 * n * m * c * k * k * out * out > 16e9:
            n //= 2
        while 2.0 * n * m * c * k * k * out * out > 16e9:
            m //= 2
        return {key: v for key, v in _conv("", weights, n, c, hw, m, k, stride, rng.random() < 0.5, rng.random() < 0.5,
                                           weights != "f32" and rng.random() < 0.3).items() if key != "name"}
    if kind == "linear":
        return {key: v for key, v in _linear("", rng.choice(["binary", "binary", "ternary"]), _log_int(rng, 1, 4096),
                                             _log_int(rng, 64, 4096), _log_int(rng, 64, 4096), rng.random() < 0.5,
                                             rng.random() < 0.5).items() if key != "name"}
    if kind == "dense":
        return {"kind": "dense", "m": _log_int(rng, 1, 2048), "k": _log_int(rng, 64, 2048),
                "n": _log_int(rng, 64, 2048), "bias": rng.random() < 0.5, "trans_b": rng.random() < 0.5}
    return {"kind": kind, "m": _log_int(rng, 1, 4096), "k": _log_int(rng, 64, 4096), "n": _log_int(rng, 64, 4096)}


# ---- inputs ------------------------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device=DEVICE)


def _signs(g, *shape):
    """BINARY bytes: 1 is +1, 0 is -1."""
    return (torch.rand(shape, generator=g, device=DEVICE) < 0.5).to(torch.uint8)


def _ternary(g, *shape):
    u = torch.rand(shape, generator=g, device=DEVICE)
    return (u >= 0.7).to(torch.int8) - (u < 0.3).to(torch.int8)


def _inputs(case, seed):
    """The tensors of a layer case, a function of the seed alone."""
    g = _generator(seed)
    kind = case["kind"]
    if kind == "conv":
        c, m, k, hw = case["c"], case["m"], case["k"], case["hw"]
        out = (hw + 2 * (k // 2) - k) // case["stride"] + 1
        x = _normal(g, case["n"], c, hw, hw)
        if case["weights"] == "ternary":
            w = _ternary(g, m, c, k, k)
        elif case["weights"] == "f32":
            w = _normal(g, m, c, k, k) * (2.0 / (c * k * k)) ** 0.5
        else:
            w = _signs(g, m, c, k, k)
        return {"x": x, "w": w, "scale": torch.rand(m, generator=g, device=DEVICE) + 0.5,
                "bias": _normal(g, m) * 0.01 if case["bias"] else None,
                "residual": _normal(g, case["n"], m, out, out) if case["residual"] else None,
                "y": torch.empty(case["n"], m, out, out, device=DEVICE)}
    m, k, n = case["m"], case["k"], case["n"]
    a = _normal(g, m, k)
    if kind == "dense":
        w = _normal(g, *((n, k) if case["trans_b"] else (k, n))) * (1.0 / k) ** 0.5
    else:
        w = _ternary(g, k, n) if case.get("weights") == "ternary" else _signs(g, k, n)
    return {"a": a, "w": w, "scale": torch.rand(n, generator=g, device=DEVICE) + 0.5,
            "bias": _normal(g, n) * 0.01 if case.get("bias") else None, "out": torch.empty(m, n, device=DEVICE)}


# ---- the models --------------------------------------------------------------------------
# A network is a list of steps (op, name, inputs, attributes); both the Session
# graph and the 64-bit evaluation below are made from it.


def _binarized(w):
    """sign(w) * mean|w| per output channel, the weights of a network trained for a binary forward."""
    flat = w.reshape(w.shape[0], -1)
    s = np.abs(flat).mean(axis=1, dtype=np.float64).astype(np.float32)
    return (np.where(flat >= 0, np.float32(1), np.float32(-1)) * s[:, None]).reshape(w.shape)


def _network(case, seed):
    rng = np.random.default_rng(int(seed))
    b = case["batch"]
    steps, inits, shapes = [], {}, {}

    def normal(shape, std):
        return rng.standard_normal(shape, dtype=np.float32) * np.float32(std)

    def conv(name, src, m, k, stride, pad, binary=True, bias=False):
        _, c, h, w = shapes[src]
        weights = normal((m, c, k, k), (2.0 / (c * k * k)) ** 0.5)
        inits[name + "_w"] = _binarized(weights) if binary else weights
        ins = [src, name + "_w"]
        if bias:
            inits[name + "_b"] = normal((m,), 0.01)
            ins.append(name + "_b")
        attrs = {"kernel_shape": [k, k], "strides": [stride, stride], "pads": [pad] * 4}
        if not binary:
            attrs["tbn_quantize"] = 0
        steps.append(("Conv", name, ins, attrs))
        shapes[name] = (b, m, (h + 2 * pad - k) // stride + 1, (w + 2 * pad - k) // stride + 1)
        return name

    def same(op, name, *src):
        steps.append((op, name, list(src), {}))
        shapes[name] = shapes[src[0]]
        return name

    def pool(name, src, k, stride, pad):
        _, c, h, w = shapes[src]
        steps.append(("MaxPool", name, [src], {"kernel_shape": [k, k], "strides": [stride, stride],
                                               "pads": [pad] * 4}))
        shapes[name] = (b, c, (h + 2 * pad - k) // stride + 1, (w + 2 * pad - k) // stride + 1)
        return name

    def head(src, classes, quantized):
        n = int(np.prod(shapes[src][1:]))
        steps.append(("Flatten", "flat", [src], {"axis": 1}))
        shapes["flat"] = (b, n)
        w = normal((n, classes), (1.0 / n) ** 0.5)
        inits["fc_w"] = np.ascontiguousarray(_binarized(w.T).T) if quantized else w
        inits["fc_b"] = normal((classes,), 0.01)
        steps.append(("Gemm", "logits", ["flat", "fc_w", "fc_b"], {} if quantized else {"tbn_quantize": 0}))
        shapes["logits"] = (b, classes)

    if case["model"] == "lenet":
        shapes["input"] = (b, 1, 28, 28)
        x = pool("pool_a", same("Relu", "act_a", conv("layer_a", "input", 6, 5, 1, 0, bias=True)), 2, 2, 0)
        x = pool("pool_b", same("Relu", "act_b", conv("layer_b", x, 16, 5, 1, 0, bias=True)), 2, 2, 0)
        head(x, 10, True)
        images = torch.rand(shapes["input"], generator=_generator(seed), device=DEVICE)
    else:
        shapes["input"] = (b, 3, 224, 224)
        x = same("Relu", "stem_act", conv("stem", "input", 64, 7, 2, 3, binary=False))
        x = pool("stem_pool", x, 3, 2, 1)
        for stage, m in enumerate((64, 128, 256, 512)):
            for block in range(2):
                pre = "s%d_%d_" % (stage, block)
                stride = 2 if stage and not block else 1
                y = same("Relu", pre + "act_a", conv(pre + "a", x, m, 3, stride, 1))
                y = conv(pre + "b", y, m, 3, 1, 1)
                skip = x if stride == 1 else conv(pre + "skip", x, m, 1, stride, 0)
                x = same("Relu", pre + "act_b", same("Add", pre + "sum", y, skip))
        steps.append(("GlobalAveragePool", "gap", [x], {}))
        shapes["gap"] = (b, shapes[x][1], 1, 1)
        head("gap", 1000, False)
        images = _normal(_generator(seed), *shapes["input"])
    return steps, inits, shapes, images


class _Memory:
    """Device memory of a framework tensor as torch.as_tensor reads it."""

    def __init__(self, t):
        self.owner = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": "<f4", "strides": None, "version": 2,
                                         "data": (t.data_ptr(), False)}


def _as_torch(t):
    return torch.as_tensor(_Memory(t), device=DEVICE)


# ---- prepare and run ---------------------------------------------------------------------


def _pack(weights, w, k, n, layout):
    k_pad, n_pad = tbn_hip.padded_dims(k, n)
    ternary = weights == "ternary"
    packed = torch.empty(n_pad * k_pad // (4 if ternary else 8), dtype=torch.uint8, device=DEVICE)
    tbn_hip.call("tbn_hip_pack_ternary" if ternary else "tbn_hip_pack_binary", w.data_ptr(), k, n, layout, k_pad,
                 n_pad, packed.data_ptr(), torch.cuda.current_stream().cuda_stream)
    return packed, k_pad, n_pad


def _bytes_of(name, *args):
    n = ctypes.c_int64()
    tbn_hip.call(name, *args, ctypes.byref(n))
    return torch.empty(max(16, n.value), dtype=torch.uint8, device=DEVICE)


def prepare(case, seed):
    stream = torch.cuda.current_stream().cuda_stream
    kind = case["kind"]
    if kind == "model":
        steps, inits, shapes, images = _network(case, seed)
        graph = _tbn.ModelGraph()
        graph.add_input("input", list(shapes["input"]))
        graph.add_output("logits", list(shapes["logits"]))
        for name, shape in shapes.items():
            graph.set_value_info(name, list(shape))
        for name, array in inits.items():
            graph.add_initializer(name, array, "float32")
        for op, name, ins, attrs in steps:
            graph.add_node(name + "_node", op, ins, [name], attrs)
        model = _tbn.TBNModel(graph)
        session = model.create_session()
        session.set_quantization(True)
        _tbn.set_current_stream(stream)
        x = _tbn.Tensor.wrap(images.data_ptr(), list(shapes["input"]), "float32", "hip")
        session.set_input("input", x)
        session.run()  # the first forward compiles the plan
        return {"case": case, "model": model, "session": session, "images": images, "x": x,
                "out": _as_torch(session.get_output_device("logits"))}

    s = _inputs(case, seed)
    s["case"], s["stream"] = case, stream
    if kind == "matmul":
        _tbn.set_current_stream(stream)
        s["ta"] = _tbn.Tensor.wrap(s["a"].data_ptr(), [case["m"], case["k"]], "float32", "hip")
        s["tw"] = _tbn.Tensor.wrap(s["w"].data_ptr(), [case["k"], case["n"]], "binary", "hip")
    elif kind in ("linear", "tbn"):
        s["packed"], s["k_pad"], s["n_pad"] = _pack(case.get("weights", "binary"), s["w"], case["k"], case["n"],
                                                    tbn_hip.LAYOUT_KN)
    elif kind == "conv":
        n, c, hw, m, k, stride = (case[v] for v in ("n", "c", "hw", "m", "k", "stride"))
        desc = s["desc"] = tbn_hip.conv_desc(n, c, hw, hw, m, k, k, stride, stride, k // 2, k // 2)
        s["flags"] = tbn_hip.EPI_RELU if case["relu"] else 0
        if case["weights"] != "f32":
            packed, k_pad, n_pad = _pack(case["weights"], s["w"], c * k * k, m, tbn_hip.LAYOUT_NK)
        if case["weights"] == "tbn":
            s["wc"] = _bytes_of("tbn_hip_tbn_conv_weights_bytes", desc)
            s["scratch"] = _bytes_of("tbn_hip_tbn_conv_scratch_bytes", desc)
            tbn_hip.call("tbn_hip_pack_tbn_conv_weights", packed.data_ptr(), k_pad, n_pad, desc, s["wc"].data_ptr(),
                         stream)
        elif case["weights"] != "f32":
            which = tbn_hip.WEIGHTS_TERNARY if case["weights"] == "ternary" else tbn_hip.WEIGHTS_BINARY
            s["which"] = which
            s["wc"] = _bytes_of("tbn_hip_conv_weights_bytes", which, desc)
            tbn_hip.call("tbn_hip_pack_conv_weights", which, packed.data_ptr(), k_pad, n_pad, desc,
                         s["wc"].data_ptr(), stream)
            # the tile of a layer shape is timed once per process, as a Session does when it compiles
            tbn_hip.call("tbn_hip_conv2d_tune_prepacked", which, s["x"].data_ptr(), desc, s["wc"].data_ptr(),
                         s["scale"].data_ptr(), 1.0, tbn_hip.ptr(s["bias"]), tbn_hip.ptr(s["residual"]), s["flags"],
                         s["y"].data_ptr(), stream)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "model":
        s["session"].set_input("input", s["x"])
        s["session"].run()
        return s["out"]
    if kind == "matmul":
        return _as_torch(_tbn.qlinear_matmul_binary(s["ta"], s["tw"], 1.0))
    if kind == "conv":
        x, y, scale = s["x"].data_ptr(), s["y"].data_ptr(), s["scale"].data_ptr()
        bias, residual = tbn_hip.ptr(s["bias"]), tbn_hip.ptr(s["residual"])
        if case["weights"] == "f32":
            tbn_hip.call("tbn_hip_conv2d_f32", x, s["desc"], s["w"].data_ptr(), bias, s["flags"], y, s["stream"])
        elif case["weights"] == "tbn":
            tbn_hip.call("tbn_hip_conv2d_tbn_prepacked", x, s["desc"], s["wc"].data_ptr(), scale, 1.0, bias, residual,
                         s["flags"], -TERNARIZE, TERNARIZE, s["scratch"].data_ptr(), y, s["stream"])
        else:
            tbn_hip.call("tbn_hip_conv2d_f32_prepacked", s["which"], x, s["desc"], s["wc"].data_ptr(), scale, 1.0,
                         bias, residual, s["flags"], y, s["stream"])
        return s["y"]
    m, k, n = case["m"], case["k"], case["n"]
    a, out, bias = s["a"].data_ptr(), s["out"].data_ptr(), tbn_hip.ptr(s["bias"])
    if kind == "dense":
        tbn_hip.call("tbn_hip_gemm_f32", a, s["w"].data_ptr(), bias, 1, m, k, n, 1.0, 1.0 if case["bias"] else 0.0, 0,
                     int(case["trans_b"]), 0, out, s["stream"])
    elif kind == "tbn":
        tbn_hip.call("tbn_hip_qlinear_matmul_binary_tbn", a, k, m, k, s["packed"].data_ptr(), s["k_pad"], n,
                     s["n_pad"], 0.75, -TERNARIZE, TERNARIZE, out, n, s["stream"])
    else:
        entry = "tbn_hip_gemm_f32_ternary" if case["weights"] == "ternary" else "tbn_hip_gemm_f32_binary"
        tbn_hip.call(entry, a, k, m, n, k, s["packed"].data_ptr(), s["k_pad"], s["n_pad"], s["scale"].data_ptr(), 1.0,
                     bias, tbn_hip.EPI_RELU if case["relu"] else 0, out, n, s["stream"])
    return s["out"]


# ---- what a pass cannot do without, and what it should give ------------------------------


def work(case):
    kind = case["kind"]
    if kind == "model":
        # fp32 input, weights (one bit each where binary) and logits; the
        # products of every layer
        layers = [(1, 6, 5, 24, 1.0 / 8), (6, 16, 5, 8, 1.0 / 8), (256, 10, 1, 1, 1.0 / 8)]
        image = 28 * 28
        if case["model"] == "resnet18":
            layers, image, c, hw = [(3, 64, 7, 112, 4.0)], 3 * 224 * 224, 64, 56
            for stage, m in enumerate((64, 128, 256, 512)):
                hw = 56 >> stage
                layers += [(c, m, 3, hw, 1.0 / 8)] + [(m, m, 3, hw, 1.0 / 8)] * 3
                layers += [(c, m, 1, hw, 1.0 / 8)] if stage else []
                c = m
            layers += [(512, 1000, 1, 1, 4.0)]
        flops = sum(2.0 * case["batch"] * c * m * k * k * hw * hw for c, m, k, hw, _ in layers)
        weights = sum(c * m * k * k * per for c, m, k, _, per in layers)
        return {"bytes": 4.0 * case["batch"] * (image + layers[-1][1]) + weights, "flops": flops}
    per = {"binary": 1.0 / 8, "tbn": 1.0 / 8, "ternary": 1.0 / 4, "f32": 4.0}
    if kind == "conv":
        out = (case["hw"] + 2 * (case["k"] // 2) - case["k"]) // case["stride"] + 1
        y = case["n"] * case["m"] * out * out
        taps = case["c"] * case["k"] ** 2
        x = case["n"] * case["c"] * case["hw"] ** 2
        return {"bytes": 4.0 * (x + y * (2 if case["residual"] else 1)) + taps * case["m"] * per[case["weights"]],
                "flops": 2.0 * y * taps}
    m, k, n = case["m"], case["k"], case["n"]
    weights = {"dense": 4.0, "matmul": 1.0, "tbn": 1.0 / 8}.get(kind) or per[case["weights"]]
    return {"bytes": 4.0 * (m * k + m * n) + k * n * weights, "flops": 2.0 * m * k * n}


def tolerance(case):
    # TBN arithmetic is exact in integers and the steps after it are fixed:
    # the same bits always
    if case["kind"] == "tbn" or case.get("weights") == "tbn":
        return "exact"
    # a network carries each layer's rounding through all that follow
    if case["kind"] == "model":
        return {"rel": 2e-6}
    # 32-bit sums in another order, up to 12800 products each: 2e-7 to 6e-7 off
    # 64 bits at the listed sizes, about 1e-6 at the longest sums
    return {"rel": 4e-6}


def _conv64(x, w, stride, pad):
    n, m, k = x.shape[0], w.shape[0], w.shape[2]
    out = (x.shape[2] + 2 * pad - k) // stride + 1
    rows = w.double().reshape(m, -1)
    y = torch.empty(n, m, out * out, dtype=torch.float64, device=x.device)
    for i in range(n):  # an image at a time keeps the columns small
        y[i] = rows @ torch.nn.functional.unfold(x[i:i + 1].double(), k, padding=pad, stride=stride)[0]
    return y.reshape(n, m, out, out)


def _ternarized(x):
    t = torch.tensor(TERNARIZE, dtype=torch.float32, device=x.device)
    return (x > t).double() - (x < -t).double()


def _model64(case, seed):
    steps, inits, shapes, images = _network(case, seed)
    quantized = {}
    env = {"input": images.double()}
    for op, name, ins, attrs in steps:
        x = env[ins[0]]
        if op == "Conv":
            w, scale = inits[ins[1]], None
            if attrs.get("tbn_quantize", 1):
                # a quantized conv's scale is the fp32 mean of |w|, summed in order
                flat = np.abs(w.reshape(w.shape[0], -1))
                mean = np.cumsum(flat, axis=1, dtype=np.float32)[:, -1] / np.float32(flat.shape[1])
                scale = torch.from_numpy(mean.astype(np.float64)).to(DEVICE)
                w = np.where(w >= 0, np.float32(1), np.float32(-1))
            y = _conv64(x, torch.from_numpy(w).to(DEVICE), attrs["strides"][0], attrs["pads"][0])
            if len(ins) > 2:
                y = y + torch.from_numpy(inits[ins[2]]).to(DEVICE).double()[None, :, None, None]
            env[name] = y if scale is None else y * scale[None, :, None, None]
        elif op == "Gemm":
            w = torch.from_numpy(inits[ins[1]]).to(DEVICE).double()
            if attrs.get("tbn_quantize", 1):
                # a quantized Gemm multiplies by the signs alone
                w = (w > 0).double() * 2 - 1
            env[name] = x @ w + torch.from_numpy(inits[ins[2]]).to(DEVICE).double()
        elif op == "MaxPool":
            env[name] = torch.nn.functional.max_pool2d(x, attrs["kernel_shape"][0], attrs["strides"][0],
                                                       attrs["pads"][0])
        elif op == "Relu":
            env[name] = x.clamp_min(0)
        elif op == "Add":
            env[name] = x + env[ins[1]]
        elif op == "GlobalAveragePool":
            env[name] = x.mean(dim=(2, 3), keepdim=True)
        else:  # Flatten
            env[name] = x.reshape(x.shape[0], -1)
    return env["logits"]


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        return _model64(case, seed)
    s = _inputs(case, seed)
    w = s["w"].double()
    if kind != "dense" and case.get("weights") not in ("ternary", "f32"):
        w = w * 2 - 1
    bias = s["bias"].double() if s["bias"] is not None else 0.0
    if kind == "conv":
        x = _ternarized(s["x"]) if case["weights"] == "tbn" else s["x"]
        y = _conv64(x, w, case["stride"], case["k"] // 2)
        if case["weights"] != "f32":
            y = y * s["scale"].double()[None, :, None, None]
        if case["bias"]:
            y = y + bias[None, :, None, None]
        if case["residual"]:
            y = y + s["residual"].double()
        return y.clamp_min(0) if case["relu"] else y
    if kind == "tbn":
        return _ternarized(s["a"]) @ w * 0.75
    y = s["a"].double() @ (w.T if case.get("trans_b") else w)
    if kind == "linear":
        y = y * s["scale"].double()
    y = y + bias
    return y.clamp_min(0) if case.get("relu") else y
