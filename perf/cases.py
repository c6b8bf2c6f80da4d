"""What a user of this framework has it do, as cases that can be timed: whole quantized networks, single convolutions,
separable pairs, fully connected and pooling layers and the conversion of camera images, through the operators of the
C ABI as the package exposes them (create once, then run on device tensors and a stream).

A case is a dict of plain values; `listed()` names the fixed ones, `draw()` makes another of the same ranges, `prepare()`
what a program has in hand before the call (weights in the operators, inputs and buffers on the GPU), `run()` one pass."""
import ctypes
import importlib
import math

import numpy as np
import torch

T = importlib.import_module("tim-vx_amd")
G = importlib.import_module("tim-vx_amd.graphs")

DTYPES = {"u8": (T.U8, torch.uint8, 1), "i8": (T.I8, torch.int8, 1), "f16": (T.F16, torch.float16, 2), "f32": (T.F32, torch.float32, 4)}
ACTS = {"none": T.ACT_NONE, "relu": T.ACT_RELU, "relu6": T.ACT_RELU6}

# Limits of the drawn cases, so that none costs more than the largest listed ones.
MOST_BYTES = 250e6
MOST_FLOPS = {"u8": 120e9, "i8": 120e9, "f16": 60e9, "f32": 8e9}


def listed():
    return [
        # One camera frame's worth of the reference's sample network: four small dependent launches.
        dict(name="lenet_u8_b1", kind="lenet", batch=1),
        # The same question for an image classifier: one image at a time, where launches and latency count.
        dict(name="mobilenet_v2_u8_b1_224", kind="mobilenet_v2", batch=1, res=224),
        # Offline classification in bulk, the throughput configuration of the repository's benchmark.
        dict(name="mobilenet_v2_u8_b64_224", kind="mobilenet_v2", batch=64, res=224),
        # The benchmark's headline layer: an early 3x3 layer of a quantized classifier, per-tensor uint8.
        dict(name="conv3x3_u8_64x56x56_b32", kind="conv", dtype="u8", batch=32, c=64, h=56, w=56, oc=64, k=3, stride=1, pad="same", act="relu6", groups=1),
        # A late layer of the same kind of network, per-channel int8: few pixels, many channels.
        dict(name="conv3x3_i8_256x14x14_b32", kind="conv", dtype="i8", batch=32, c=256, h=14, w=14, oc=256, k=3, stride=1, pad="same", act="relu", groups=1),
        # A half-precision model's middle layer on an odd plane (27 columns) with a wider window.
        dict(name="conv5x5_f16_96x27x27_b16", kind="conv", dtype="f16", batch=16, c=96, h=27, w=27, oc=256, k=5, stride=1, pad="same", act="relu", groups=1),
        # A model that has not been quantized yet, a down-sampling layer in single precision.
        dict(name="conv3x3_f32_32x112x112_b4_s2", kind="conv", dtype="f32", batch=4, c=32, h=112, w=112, oc=64, k=3, stride=2, pad="same", act="relu", groups=1),
        # MobileNetV1's first depthwise + pointwise block, per-channel int8 (the benchmark's third configuration).
        dict(name="separable_i8_112x112x32to64_b32", kind="separable", dtype="i8", batch=32, c=32, h=112, w=112, oc=64, k=3, stride=1),
        # The benchmark's large fully connected layer: many rows at once, bound by the matrix cores.
        dict(name="fc_i8_8192x4096x4096", kind="fc", dtype="i8", m=8192, k=4096, n=4096),
        # A half-precision hidden layer for a small batch: bound by reading the weights.
        dict(name="fc_f16_16x4096x4096", kind="fc", dtype="f16", m=16, k=4096, n=4096),
        # The pooling behind a first layer, SAME padding as converters emit it.
        dict(name="maxpool3x3s2_u8_112x112x64_b32", kind="pool", dtype="u8", type="max", batch=32, c=64, h=112, w=112, k=3, stride=2, pad="same"),
        # Float images as a camera pipeline or an NHWC model hands them over: quantized, then reordered to planes.
        dict(name="ingest_u8_224x224x3_b32", kind="ingest", to="u8", batch=32, c=3, h=224, w=224),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _channels(rng, lo, hi):
    """Channel counts: mostly multiples of 8 or 16 as networks have them, one in four anything."""
    n = _log(rng, lo, hi)
    if rng.random() < 0.25:
        return n
    step = 16 if n >= 64 else 8
    return max(step, (n + step // 2) // step * step)


def _plane(rng, lo, hi):
    """Height and width: square planes mostly."""
    h = _log(rng, lo, hi)
    return (h, h) if rng.random() < 0.75 else (h, min(hi, max(lo, int(round(h * rng.uniform(0.5, 2.0))))))


def _dtype(rng):
    return rng.choice(("u8", "u8", "u8", "i8", "i8", "i8", "f16", "f16", "f32"))


def _draw_once(rng):
    kind = rng.choice(("lenet", "mobilenet_v2", "conv", "conv", "conv", "conv", "separable", "separable", "fc", "fc", "pool", "ingest"))
    if kind == "lenet":
        return dict(kind=kind, batch=_log(rng, 1, 256))
    if kind == "mobilenet_v2":
        return dict(kind=kind, batch=_log(rng, 1, 64), res=32 * rng.randint(3, 7))
    if kind == "conv":
        h, w = _plane(rng, 7, 160)
        # a first layer has 1 or 3 channels; the others 8 to 512
        first = rng.random() < 0.15
        c = rng.choice((1, 3)) if first else _channels(rng, 8, 512)
        oc = _channels(rng, 8, 96) if first else _channels(rng, 8, 512)
        groups = 1
        if not first and rng.random() < 0.1:
            groups = rng.choice((2, 4))
            c, oc = -(-c // groups) * groups, -(-oc // groups) * groups
        k = rng.choice((1, 1, 3, 3, 3, 3, 5, 7)) if min(h, w) >= 7 else 3
        return dict(kind=kind, dtype=_dtype(rng), batch=_log(rng, 1, 64), c=c, h=h, w=w, oc=oc, k=k, stride=rng.choice((1, 1, 1, 2)),
                    pad=rng.choice(("same", "same", "same", "valid")), act=rng.choice(("none", "relu", "relu6")), groups=groups)
    if kind == "separable":
        h, w = _plane(rng, 7, 160)
        return dict(kind=kind, dtype=_dtype(rng), batch=_log(rng, 1, 64), c=_channels(rng, 8, 512), h=h, w=w, oc=_channels(rng, 8, 512),
                    k=rng.choice((3, 3, 3, 5)), stride=rng.choice((1, 1, 2)))
    if kind == "fc":
        return dict(kind=kind, dtype=_dtype(rng), m=_log(rng, 1, 8192), k=_channels(rng, 64, 4096), n=_log(rng, 10, 4096))
    if kind == "pool":
        h, w = _plane(rng, 7, 160)
        k, stride = rng.choice(((2, 2), (3, 2), (3, 1), (7, 7), (0, 1)))  # 0: the whole plane
        return dict(kind=kind, dtype=_dtype(rng), type="avg" if k == 0 else rng.choice(("max", "max", "avg")), batch=_log(rng, 1, 64),
                    c=_channels(rng, 8, 512), h=h, w=w, k=k, stride=stride, pad="same" if k == 3 and rng.random() < 0.5 else "valid")
    h, w = _plane(rng, 16, 320)
    return dict(kind=kind, to=rng.choice(("u8", "u8", "i8", "f16")), batch=_log(rng, 1, 64), c=rng.choice((1, 3, 3, 3, 4, _channels(rng, 8, 256))), h=h, w=w)


def draw(rng):
    while True:
        case = _draw_once(rng)
        if case["kind"] in ("lenet", "mobilenet_v2"):
            return case
        w = work(case)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS.get(case.get("dtype"), 8e9):
            return case


# ---- shapes ----

def _window(case):
    """(output height, output width, pad top, pad left) of a windowed layer."""
    k, s = case["k"], case["stride"]
    kh, kw = (k, k) if k else (case["h"], case["w"])
    if case.get("pad", "same") == "valid":
        return (case["h"] - kh) // s + 1, (case["w"] - kw) // s + 1, 0, 0
    oh, top, _ = G.same_pad(case["h"], kh, s)
    ow, left, _ = G.same_pad(case["w"], kw, s)
    return oh, ow, top, left


def _graph(case, seed):
    if case["kind"] == "lenet":
        return G.lenet_random(batch=case["batch"], seed=seed)
    return G.mobilenet_v2(batch=case["batch"], res=case["res"], seed=seed)


def _size(shape):
    return int(np.prod(shape))


def work(case):
    kind = case["kind"]
    if kind in ("lenet", "mobilenet_v2"):
        g = _graph(case, 0)
        width = {"UINT8": 1, "INT32": 4, "FLOAT32": 4}
        return {"bytes": sum(_size(t["shape"]) * width[t["dtype"]] for t in g["tensors"] if t["attr"] != "TRANSIENT"), "flops": 2 * G.mac_count(g)}
    if kind == "fc":
        m, k, n, e = case["m"], case["k"], case["n"], DTYPES[case["dtype"]][2]
        return {"bytes": e * (m * k + k * n + m * n) + 4 * n, "flops": 2 * m * k * n}
    pixels_in = case["batch"] * case["h"] * case["w"]
    if kind == "ingest":
        return {"bytes": pixels_in * case["c"] * (4 + DTYPES[case["to"]][2]), "flops": 2 * pixels_in * case["c"]}
    e = DTYPES[case["dtype"]][2]
    oh, ow, _, _ = _window(case)
    pixels_out = case["batch"] * oh * ow
    if kind == "pool":
        taps = case["k"] ** 2 if case["k"] else case["h"] * case["w"]
        return {"bytes": e * case["c"] * (pixels_in + pixels_out), "flops": pixels_out * case["c"] * taps}
    if kind == "separable":
        c, oc, taps = case["c"], case["oc"], case["k"] ** 2
        return {"bytes": e * (pixels_in * c + pixels_out * oc + c * taps + c * oc) + 4 * (c + oc), "flops": 2 * pixels_out * c * (taps + oc)}
    c, oc, reduction = case["c"], case["oc"], case["k"] ** 2 * case["c"] // case["groups"]
    return {"bytes": e * (pixels_in * c + pixels_out * oc + oc * reduction) + 4 * oc, "flops": 2 * pixels_out * oc * reduction}


def tolerance(case):
    if case["kind"] == "lenet":
        return {"rel": 1e-5}  # the Softmax behind exact codes
    if case.get("type") == "max":
        return "exact"
    return {"f16": {"rel": 1e-3}, "f32": {"rel": 1e-5}}.get(case.get("dtype"), "exact")


# ---- inputs, weights and operators ----

def _input(gen, dtype, n):
    """Activations: codes over their whole range, floats normally distributed."""
    if dtype in ("u8", "i8"):
        lo, hi = (0, 256) if dtype == "u8" else (-128, 128)
        return torch.randint(lo, hi, (n,), dtype=DTYPES[dtype][1], device="cuda", generator=gen)
    return torch.randn(n, dtype=torch.float32, device="cuda", generator=gen).to(DTYPES[dtype][1])


def _empty(dtype, n):
    return torch.empty(n, dtype=DTYPES[dtype][1], device="cuda")


class _Quant:
    """Quantization and weights of one layer: uint8 per tensor, int8 per channel or floating point. The output scale
    spreads the results over the codes, as calibration does."""

    def __init__(self, rng, dtype, reduction, channels, in_scale=0.05, in_zp=None, act="none"):
        n = reduction * channels
        self.dtype, self.scales, self.w_zp = dtype, None, 0
        self.in_scale = self.out_scale = self.w_scale = 1.0
        self.in_zp = self.out_zp = 0
        if dtype in ("u8", "i8"):
            self.in_scale = in_scale
            self.in_zp = (128 if dtype == "u8" else 0) if in_zp is None else in_zp
            spread = 74.0 * 74.0 * math.sqrt(reduction) * in_scale * 0.01
            self.out_scale = spread / (100.0 if act != "none" else 40.0)
            self.out_zp = (0 if dtype == "u8" else -128) if act != "none" else (128 if dtype == "u8" else 0)
            self.bias = rng.integers(-4096, 4097, channels).astype(np.int32)
        if dtype == "u8":
            self.w_scale, self.w_zp = 0.01, 120
            self.weights = rng.integers(0, 256, n, dtype=np.uint8)
        elif dtype == "i8":
            self.scales = (0.01 * np.exp(rng.uniform(-0.7, 0.7, channels))).astype(np.float32)
            self.weights = rng.integers(-128, 128, n, dtype=np.int8)
        else:
            np_type = np.float16 if dtype == "f16" else np.float32
            self.weights = (rng.standard_normal(n, dtype=np.float32) / math.sqrt(reduction)).astype(np_type)
            self.bias = (0.1 * rng.standard_normal(channels)).astype(np.float32)

    def fill(self, d):
        d.in_dtype = d.w_dtype = d.out_dtype = DTYPES[self.dtype][0]
        d.in_scale, d.in_zp, d.w_scale, d.w_zp = self.in_scale, self.in_zp, self.w_scale, self.w_zp
        if self.scales is not None:
            d.w_scales = self.scales.ctypes.data_as(ctypes.POINTER(ctypes.c_float))
        d.out_scale, d.out_zp = self.out_scale, self.out_zp


def _conv_desc(batch, c, h, w, oc, oh, ow, k, stride, top, left, act, multiplier=0, groups=1):
    d = T.Conv2dDesc()
    d.in_w, d.in_h, d.in_c, d.batch = w, h, c, batch
    d.k_w = d.k_h = k
    d.out_w, d.out_h, d.out_c = ow, oh, oc
    d.stride_w = d.stride_h = stride
    d.dilation_w = d.dilation_h = 1
    d.pad_left, d.pad_top, d.multiplier, d.groups = left, top, multiplier, groups
    d.activation = ACTS[act]
    return d


def _create(make, *args):
    """The fused operator, or None where the library has none for these shapes and the parts are to be made one by one."""
    try:
        return make(*args)
    except T.TvxError as e:
        if e.status != T.E_UNSUPPORTED:
            raise
        return None


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator("cuda").manual_seed(seed)
    state = {"stream": torch.cuda.current_stream().cuda_stream}
    return globals()["_prepare_" + ("network" if case["kind"] in ("lenet", "mobilenet_v2") else case["kind"])](case, seed, rng, gen, state)


def run(state):
    stream = state["stream"]
    for op, in0, in1, out in state["steps"]:
        op.run(in0, in1, out, stream)
    return state["out"]


def _prepare_conv(case, seed, rng, gen, state):
    oh, ow, top, left = _window(case)
    c, oc, k, n = case["c"], case["oc"], case["k"], case["batch"]
    q = _Quant(rng, case["dtype"], k * k * c // case["groups"], oc, act=case["act"])
    d = _conv_desc(n, c, case["h"], case["w"], oc, oh, ow, k, case["stride"], top, left, case["act"], groups=case["groups"])
    q.fill(d)
    op = T.conv2d_create(d, q.weights, q.bias)
    x, y = _input(gen, case["dtype"], n * c * case["h"] * case["w"]), _empty(case["dtype"], n * oc * oh * ow)
    return dict(state, steps=[(op, x, None, y)], out=y)


def _prepare_separable(case, seed, rng, gen, state):
    """A depthwise convolution and the 1x1 convolution behind it: one operator where the library merges them, else two."""
    oh, ow, top, left = _window(case)
    c, oc, k, n, dtype = case["c"], case["oc"], case["k"], case["batch"], case["dtype"]
    qd = _Quant(rng, dtype, k * k, c)
    qp = _Quant(rng, dtype, c, oc, in_scale=qd.out_scale, in_zp=qd.out_zp, act="relu6")
    if dtype in ("u8", "i8"):
        qp.out_scale = 6.0 / 255.0
    dw = _conv_desc(n, c, case["h"], case["w"], c, oh, ow, k, case["stride"], top, left, "none", multiplier=1)
    pw = _conv_desc(n, c, oh, ow, oc, oh, ow, 1, 1, 0, 0, "relu6")
    qd.fill(dw)
    qp.fill(pw)
    x, y = _input(gen, dtype, n * c * case["h"] * case["w"]), _empty(dtype, n * oc * oh * ow)
    both = _create(T.conv2d_dw_pw_create, dw, qd.weights, qd.bias, pw, qp.weights, qp.bias)
    if both:
        return dict(state, steps=[(both, x, None, y)], out=y)
    mid = _empty(dtype, n * c * oh * ow)
    steps = [(T.conv2d_create(dw, qd.weights, qd.bias), x, None, mid), (T.conv2d_create(pw, qp.weights, qp.bias), mid, None, y)]
    return dict(state, steps=steps, out=y)


def _prepare_fc(case, seed, rng, gen, state):
    m, k, n = case["m"], case["k"], case["n"]
    q = _Quant(rng, case["dtype"], k, n)
    d = T.FcDesc()
    d.m, d.k, d.n = m, k, n
    q.fill(d)
    op = T.fully_connected_create(d, q.weights, q.bias)
    x, y = _input(gen, case["dtype"], m * k), _empty(case["dtype"], m * n)
    return dict(state, steps=[(op, x, None, y)], out=y)


def _prepare_pool(case, seed, rng, gen, state):
    oh, ow, top, left = _window(case)
    d = T.Pool2dDesc()
    d.in_w, d.in_h, d.channels, d.batch = case["w"], case["h"], case["c"], case["batch"]
    d.out_w, d.out_h = ow, oh
    d.k_w, d.k_h = (case["k"], case["k"]) if case["k"] else (case["w"], case["h"])
    d.stride_w = d.stride_h = case["stride"]
    d.pad_left, d.pad_top = left, top
    d.pool_type = T.POOL_MAX if case["type"] == "max" else T.POOL_AVG_ANDROID if case["pad"] == "same" else T.POOL_AVG
    d.dtype = DTYPES[case["dtype"]][0]
    d.in_scale = d.out_scale = 0.05
    d.in_zp = d.out_zp = {"u8": 3, "i8": -4}.get(case["dtype"], 0)
    op = T.pool2d_create(d)
    planes = case["batch"] * case["c"]
    x, y = _input(gen, case["dtype"], planes * case["h"] * case["w"]), _empty(case["dtype"], planes * oh * ow)
    return dict(state, steps=[(op, x, None, y)], out=y)


def _prepare_ingest(case, seed, rng, gen, state):
    """Float images, channels fastest ({C, W, H, N}), to a network's input tensor ({W, H, C, N})."""
    to, dims = case["to"], [case["c"], case["w"], case["h"], case["batch"]]
    count = _size(dims)
    cd = T.ConvertDesc()
    cd.count, cd.in_dtype, cd.in_scale, cd.in_zp = count, T.F32, 1.0, 0
    cd.out_dtype, cd.out_scale, cd.out_zp = DTYPES[to][0], 1.0 if to == "f16" else 1.0 / 128, {"u8": 128}.get(to, 0)
    td = T.TransposeDesc()
    td.rank, td.elem_bytes = 4, DTYPES[to][2]
    for i, (size, source) in enumerate(zip(dims, (1, 2, 0, 3))):
        td.in_dims[i], td.perm[i] = size, source
    x = torch.rand(count, dtype=torch.float32, device="cuda", generator=gen) * 2.0 - 1.0
    mid, y = _empty(to, count), _empty(to, count)
    return dict(state, steps=[(T.convert_create(cd), x, None, mid), (T.transpose_create(td), mid, None, y)], out=y)


# ---- whole networks: a graph description to a sequence of operators ----

class _Planner:
    """Turns a graph description into operators in order: an activation goes into the layer in front of it, chains that
    the library merges become one operator (it says where it has none), everything else is an operator of its own."""

    def __init__(self, graph, gen):
        self.tensors = {t["id"]: t for t in graph["tensors"]}
        self.output = graph["output"]
        self.nodes = self._with_activations(graph["ops"])
        self.buffers = {}
        for t in graph["tensors"]:
            if t["attr"] == "INPUT":
                self.buffers[t["id"]] = _input(gen, "u8", _size(t["shape"]))

    def _with_activations(self, ops):
        self.readers = {}
        for o in ops:
            for i in o["inputs"]:
                self.readers[i] = self.readers.get(i, 0) + 1
        nodes = []
        for o in ops:
            node = dict(o, act=T.ACT_NONE, out=o["outputs"][0])
            if o["kind"] in ("RELU", "RELU6") and nodes[-1]["out"] == o["inputs"][0] and self.readers[o["inputs"][0]] == 1:
                nodes[-1].update(act=T.ACT_RELU if o["kind"] == "RELU" else T.ACT_RELU6, out=node["out"])
            else:
                nodes.append(node)
        return nodes

    def _q(self, tid):
        quant = self.tensors[tid]["quant"]
        return quant["scales"][0], quant["zero_points"][0]

    def _conv(self, node):
        a = node["attrs"]
        w, h, c, n = self.tensors[node["inputs"][0]]["shape"]
        ow, oh, oc, _ = self.tensors[node["out"]]["shape"]
        left, top = (0, 0) if a["pad_type"] == "VALID" else (a["pad"][0], a["pad"][2])
        d = _conv_desc(n, c, h, w, oc, oh, ow, a["ksize"][0], a["stride"][0], top, left, "none", multiplier=a["multiplier"])
        d.activation = node["act"]
        self._types(d, node)
        return d, self.tensors[node["inputs"][1]]["data"], self.tensors[node["inputs"][2]]["data"]

    def _types(self, d, node):
        d.in_dtype = d.w_dtype = d.out_dtype = T.U8
        (d.in_scale, d.in_zp), (d.w_scale, d.w_zp) = self._q(node["inputs"][0]), self._q(node["inputs"][1])
        d.out_scale, d.out_zp = self._q(node["out"])

    def _fc(self, node):
        d = T.FcDesc()
        d.k, d.n = self.tensors[node["inputs"][1]]["shape"]
        d.m = _size(self.tensors[node["inputs"][0]]["shape"]) // d.k
        d.activation = node["act"]
        self._types(d, node)
        return d, self.tensors[node["inputs"][1]]["data"], self.tensors[node["inputs"][2]]["data"]

    def _add(self, node):
        d = T.EltwiseDesc()
        d.count, d.dtype = _size(self.tensors[node["out"]]["shape"]), T.U8
        (d.a_scale, d.a_zp), (d.b_scale, d.b_zp) = self._q(node["inputs"][0]), self._q(node["inputs"][1])
        d.out_scale, d.out_zp = self._q(node["out"])
        return d

    def _pool(self, node):
        a, d = node["attrs"], T.Pool2dDesc()
        d.in_w, d.in_h, d.channels, d.batch = self.tensors[node["inputs"][0]]["shape"]
        d.out_w, d.out_h = self.tensors[node["out"]]["shape"][:2]
        (d.k_w, d.k_h), (d.stride_w, d.stride_h) = a["ksize"], a["stride"]
        d.pool_type, d.dtype = T.POOL_MAX if a["pool_type"] == "MAX" else T.POOL_AVG, T.U8
        (d.in_scale, d.in_zp), (d.out_scale, d.out_zp) = self._q(node["inputs"][0]), self._q(node["out"])
        return d

    def _softmax(self, node):
        d = T.SoftmaxDesc()
        d.channels, d.rows = self.tensors[node["inputs"][0]]["shape"]
        d.beta, d.in_dtype, d.inner = node["attrs"]["beta"], T.U8, 1
        d.in_scale, d.in_zp = self._q(node["inputs"][0])
        return d

    def _kinds(self, i):
        """The kinds of the chain that begins at node i: every further node reads the result before it, which nothing else reads."""
        kinds = []
        for j in range(i, min(i + 4, len(self.nodes))):
            node = self.nodes[j]
            if j > i and (self.nodes[j - 1]["out"] not in node["inputs"] or self.readers[self.nodes[j - 1]["out"]] != 1):
                break
            kinds.append(node["kind"] if node["kind"] != "CONV2D" else "DW" if node["attrs"]["multiplier"] else "PW" if node["attrs"]["ksize"][0] == 1 else "CONV")
        return kinds

    def _chains(self, i):
        """(nodes taken, operator, residual input) of every way to make node i, the longest merged chain first."""
        kinds, nodes = self._kinds(i), self.nodes[i:i + 4]

        def residual(at):
            """(the Add, which operand of it the chain is, the other operand)"""
            ins, mine = nodes[at]["inputs"], nodes[at - 1]["out"]
            return (self._add(nodes[at]), 1, ins[1]) if ins[0] == mine else (self._add(nodes[at]), 2, ins[0])

        for chain, make in ((["PW", "DW", "PW"], T.mbconv_create), (["DW", "PW"], T.conv2d_dw_pw_create)):
            n = len(chain)
            if kinds[:n] == chain:
                parts = [p for node in nodes[:n] for p in self._conv(node)]
                if kinds[n:n + 1] == ["ADD"]:
                    add, operand, other = residual(n)
                    yield n + 1, _create(make, *parts, add, operand), other
                yield n, _create(make, *parts), None
        if kinds[:2] in (["PW", "ADD"], ["CONV", "ADD"]):
            (d, w, b), (add, operand, other) = self._conv(nodes[0]), residual(1)
            yield 2, _create(T.conv2d_add_create, d, add, operand, w, b), other
        if kinds[:2] == ["CONV", "POOL"]:
            d, w, b = self._conv(nodes[0])
            yield 2, _create(T.conv2d_pool_create, d, self._pool(nodes[1]), w, b), None
        if kinds[:2] == ["FCL", "SOFTMAX"]:
            d, w, b = self._fc(nodes[0])
            yield 2, _create(T.fully_connected_softmax_create, d, self._softmax(nodes[1]), w, b), None
        node = nodes[0]
        if node["kind"] == "CONV2D":
            yield 1, T.conv2d_create(*self._conv(node)), None
        elif node["kind"] == "FCL":
            yield 1, T.fully_connected_create(*self._fc(node)), None
        elif node["kind"] == "ADD":
            yield 1, T.add_create(self._add(node)), node["inputs"][1]
        elif node["kind"] == "POOL":
            yield 1, T.pool2d_create(self._pool(node)), None
        else:
            yield 1, T.softmax_create(self._softmax(node)), None

    def steps(self):
        got, i = [], 0
        while i < len(self.nodes):
            taken, op, other = next(c for c in self._chains(i) if c[1] is not None)
            out = self.tensors[self.nodes[i + taken - 1]["out"]]
            y = self.buffers[out["id"]] = _empty("f32" if out["dtype"] == "FLOAT32" else "u8", _size(out["shape"]))
            got.append((op, self.buffers[self.nodes[i]["inputs"][0]], None if other is None else self.buffers[other], y))
            i += taken
        return got


def _prepare_network(case, seed, rng, gen, state):
    planner = _Planner(_graph(case, seed), gen)
    return dict(state, steps=planner.steps(), out=planner.buffers[planner.output])
