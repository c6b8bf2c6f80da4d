"""The tim::vx C++ API end to end: graphs are built by the tvx_graph_runner tool through
Context / Graph / Tensor / ops::* exactly as an application would, compiled and run by the
C++ runtime on the GPU, and compared with the reference's golden vectors and the oracle."""
import copy
import importlib
import os

import numpy as np
import pytest

import tvx_case as TC

GF = importlib.import_module("tim-vx_amd.graphfile")
GRAPHS = importlib.import_module("tim-vx_amd.graphs")
HERE = os.path.dirname(os.path.abspath(__file__))


def _lenet_data():
    z = np.load(os.path.join(HERE, "golden", "lenet_asymu8.npz"))
    return z["weights"], z["input"]


def _named_cases():
    out = []
    for _, c in TC.all_cases():
        c = dict(c)
        c["test"] = "%s#%d" % (c["test"], c["index"])
        out.append(c)
    return out


# --------------------------------------------------------------------------- CPU side
def test_runner_is_built():
    assert os.path.exists(GF.RUNNER), "tvx_graph_runner missing: run tim-vx_amd/build.py"


def test_graph_file_round_trip(tmp_path):
    """The writer emits one record per tensor / operator and the blob holds every datum."""
    w, x = _lenet_data()
    g = GRAPHS.lenet_asymu8(w, x)
    txt, blob = tmp_path / "g.txt", tmp_path / "g.bin"
    GF.write_graphs([g], str(txt), str(blob))
    lines = txt.read_text().splitlines()
    assert sum(l.startswith("t ") for l in lines) == len(g["tensors"])
    assert sum(l.startswith("op ") for l in lines) == len(g["ops"])
    assert blob.stat().st_size == 432820 + 784


def test_lenet_oracle_classifies_the_sample_digit(oracle):
    """The reference's sample image is a hand-written zero; the sample prints a top-5 and
    holds no expected numbers, so the class is what can be pinned."""
    w, x = _lenet_data()
    prob = oracle.run_graph(GRAPHS.lenet_asymu8(w, x))
    assert prob.shape == (10,) and int(np.argmax(prob)) == 0 and prob[0] > 0.99
    assert abs(float(prob.sum()) - 1.0) < 1e-5


def test_mobilenet_description_is_well_formed():
    g = GRAPHS.mobilenet_v2(batch=1, res=224)
    kinds = [o["kind"] for o in g["ops"]]
    assert kinds.count("CONV2D") == 52 and kinds.count("ADD") == 10 and kinds.count("FCL") == 1
    assert GRAPHS.mac_count(g) == 300774272  # MobileNetV2-1.0 at 224: ~300 M multiply-accumulates


def _has_gpu():
    import torch
    return torch.cuda.is_available()


def test_runtime_without_gpu_refuses_to_compile(tmp_path):
    """No CPU execution path: with no device, Compile() returns false and says why."""
    if _has_gpu():
        pytest.skip("a GPU is present")
    case = _named_cases()[0]
    res, info, log = GF.run_graphs([case], str(tmp_path))
    assert res == [None] and info[case["test"]]["fail"] == "compile"
    assert "no GPU" in log


def test_verification_errors_are_reported(tmp_path):
    """Host-side verification runs before any device work (reference behaviour: Compile()
    returns false, vsi_nn_VerifyGraph logs): a bias scale that is not input*weight scale and
    an unsupported dtype pairing."""
    base = next(c for c in _named_cases() if c["test"].startswith("Conv2d.shape_4_2_1_2_uint8_QuantizedTest1"))
    bad_bias = copy.deepcopy(base)
    bad_bias["test"] = "bad_bias_scale"
    bt = {t["id"]: t for t in bad_bias["tensors"]}[bad_bias["ops"][0]["inputs"][2]]
    bt["quant"]["scales"] = [bt["quant"]["scales"][0] * 1.5]
    bad_pair = copy.deepcopy(base)
    bad_pair["test"] = "bad_dtype_pair"
    wt = {t["id"]: t for t in bad_pair["tensors"]}[bad_pair["ops"][0]["inputs"][1]]
    wt["dtype"] = "FLOAT32"
    wt["quant"] = GF.NO_QUANT
    res, info, log = GF.run_graphs([bad_bias, bad_pair], str(tmp_path))
    assert res == [None, None]
    assert info["bad_bias_scale"]["fail"] == "compile" and info["bad_dtype_pair"]["fail"] == "compile"
    assert "bias scale" in log and "data type not support" in log


# --------------------------------------------------------------------------- GPU side
@pytest.mark.gpu
def test_every_reference_golden_through_the_cpp_api(tmp_path):
    cases = _named_cases()
    res, info, log = GF.run_graphs(cases, str(tmp_path))
    bad = []
    for c, out in zip(cases, res):
        if out is None:
            bad.append((c["test"], info.get(c["test"])))
        elif not TC.matches(c, out):
            bad.append((c["test"], out[:8], TC.golden_of(c)[:8]))
    assert not bad, (bad[:5], log[-2000:])


@pytest.mark.gpu
def test_every_reference_golden_through_the_platform_api(tmp_path):
    """The same graphs as executables of the platform API (include/tim/vx/platform/platform.h:56-145,
    samples/multi_device/multi_device_demo.cc:48-91): IDevice::Enumerate -> CreateExecutor ->
    Compile(graph) -> AllocateTensor / SetInput / SetOutput -> Submit -> Trigger. The layout-inference
    source graphs go in as they are: the executable resolves layouts when it rebuilds the graph."""
    cases = _named_cases()
    for c in cases:
        c["platform"] = True
        c["layout_inference"] = False
    res, info, log = GF.run_graphs(cases, str(tmp_path))
    bad = []
    for c, out in zip(cases, res):
        if out is None:
            bad.append((c["test"], info.get(c["test"])))
        elif not TC.matches(c, out):
            bad.append((c["test"], out[:8], TC.golden_of(c)[:8]))
    assert not bad, (bad[:5], log[-2000:])


@pytest.mark.gpu
def test_every_reference_golden_through_clone(tmp_path):
    """The same graphs with every operator created in a second graph and cloned into the one that runs
    (Operation::Clone, include/tim/vx/operation.h:46): Conv2d, Conv1d, GroupedConv2d, GroupedConv1d, DeConv2d,
    DeConv1d, FullyConnected, Pool2d, Softmax, Transpose and DataConvert each carry their attributes over."""
    cases = [c for c in _named_cases() if not c.get("layout_inference")]
    for c in cases:
        c["clone"] = True
    res, info, log = GF.run_graphs(cases, str(tmp_path))
    bad = []
    for c, out in zip(cases, res):
        if out is None:
            bad.append((c["test"], info.get(c["test"])))
        elif not TC.matches(c, out):
            bad.append((c["test"], out[:8], TC.golden_of(c)[:8]))
    assert not bad, (bad[:5], log[-2000:])


@pytest.mark.gpu
def test_lenet_sample_graph(tmp_path, oracle):
    w, x = _lenet_data()
    g = GRAPHS.lenet_asymu8(w, x)
    logits = copy.deepcopy(g)  # same graph cut before the softmax: the uint8 logits
    logits["test"] = "lenet_logits"
    logits["ops"] = logits["ops"][:-1]
    logits["tensors"] = logits["tensors"][:-1]
    logits["tensors"][15]["attr"] = "OUTPUT"
    logits["output"] = 15
    batched = GRAPHS.lenet_asymu8(w, x, batch=16)
    res, info, log = GF.run_graphs([g, logits, batched], str(tmp_path), env={"VSI_NN_LOG_LEVEL": "3"})
    assert all(r is not None for r in res), (info, log[-2000:])
    assert np.array_equal(res[1], oracle.run_graph(logits))  # bit-exact
    ref = oracle.run_graph(g)
    assert np.allclose(res[0], ref, rtol=0, atol=1e-6) and int(np.argmax(res[0])) == 0
    assert np.allclose(res[2].reshape(16, 10), ref[None, :], rtol=0, atol=1e-6)
    # FullyConnected + Relu through a single-consumer TRANSIENT tensor is fused: no separate
    # activation kernel appears in the plan
    plan = [l for l in log.splitlines() if "uid" in l and "->" in l]
    assert plan and not any("RELU" in l for l in plan), plan
    # convolution + max pooling and FullyConnected + Softmax through such tensors run as one kernel each: the
    # sample's nine operators are four launches (five where the graph ends with the logits)
    kernels = [l.split("(")[-1].rstrip(")") for l in plan]
    assert kernels[:4] == ["conv2d_im2col_maxpool_i8", "conv2d_igemm_maxpool_i8", "fc_generic", "fc_softmax_i8"], kernels
    assert kernels[4:8] == ["conv2d_im2col_maxpool_i8", "conv2d_igemm_maxpool_i8", "fc_generic", "fc_generic"], kernels
    assert len(kernels) == 12
    # ... and give the bytes of the operators run one by one
    apart, _, log2 = GF.run_graphs([g, batched], str(tmp_path / "apart"), env={"VSI_NN_LOG_LEVEL": "3", "TVX_NO_POOL_FUSION": "1"})
    assert len([l for l in log2.splitlines() if "uid" in l and "->" in l]) == 14
    assert np.array_equal(apart[0], res[0]) and np.array_equal(apart[1], res[2])


@pytest.mark.gpu
@pytest.mark.parametrize("lock", [True, False], ids=["one_mutex", "concurrent"])
def test_two_threads_build_compile_and_run_lenet(tmp_path, oracle, lock):
    """Two threads, each with a context of its own, build, compile and run LeNet (batch 1 and batch 16): one after
    the other under one mutex, as the reference's multi-thread sample does
    (samples/multi_thread_test/multi_thread_test.cc:100,330-372), and without the mutex. Every thread's bytes must
    be the single-threaded ones, bit for bit the oracle's."""
    w, x = _lenet_data()
    g = GRAPHS.lenet_asymu8(w, x)
    logits = copy.deepcopy(g)  # cut before the softmax: the uint8 logits
    logits["test"] = "lenet_logits"
    logits["ops"] = logits["ops"][:-1]
    logits["tensors"] = logits["tensors"][:-1]
    logits["tensors"][15]["attr"] = "OUTPUT"
    logits["output"] = 15
    batched = GRAPHS.lenet_random(batch=16)
    graphs = [g, logits, batched]
    single, info, log = GF.run_graphs(graphs, str(tmp_path / "single"))
    threaded, info_t, log_t = GF.run_graphs(graphs, str(tmp_path / "threads"), threads=2, lock=lock)
    assert all(r is not None for r in single) and all(r is not None for r in threaded), (info, info_t, log_t[-2000:])
    for a, b in zip(single, threaded):
        assert np.array_equal(a, b)
    assert np.array_equal(threaded[1], oracle.run_graph(logits))
    assert int(np.argmax(threaded[0])) == 0


@pytest.mark.gpu
def test_transpose_feeds_a_convolution(tmp_path, oracle):
    """A channel-fastest {C, W, H, N} image brought to WHCN by Transpose{1, 2, 0, 3} (the permute
    layout inference puts in front of an NHWC model, src/tim/transform/layout_inference.cc), then a
    3x3 convolution; the output goes back to channel-fastest through Transpose{2, 0, 1, 3}."""
    rng = np.random.default_rng(5)
    c, w, h, n, oc = 8, 12, 10, 2, 16
    q = GF.asym
    x = rng.integers(0, 256, c * w * h * n, dtype=np.uint8)
    wt = rng.integers(0, 256, 3 * 3 * c * oc, dtype=np.uint8)
    bias = rng.integers(-500, 500, oc, dtype=np.int32)
    T = GF.tensor
    g = {"test": "transpose_conv_transpose", "output": 6, "tensors": [
        T(0, "UINT8", "INPUT", [c, w, h, n], q(0.5, 128), x),
        T(1, "UINT8", "TRANSIENT", [w, h, c, n], q(0.5, 128)),
        T(2, "UINT8", "CONSTANT", [3, 3, c, oc], q(0.25, 120), wt),
        T(3, "INT32", "CONSTANT", [oc], q(0.125, 0), bias),
        T(4, "UINT8", "TRANSIENT", [w, h, oc, n], q(64.0, 100)),
        T(6, "UINT8", "OUTPUT", [oc, w, h, n], q(64.0, 100))],
        "ops": [GF.op("TRANSPOSE", [0], [1], perm=[1, 2, 0, 3]),
                GF.op("CONV2D", [1, 2, 3], [4], pad_type="AUTO", pad=[1, 1, 1, 1], ksize=[3, 3], weights=oc),
                GF.op("TRANSPOSE", [4], [6], perm=[2, 0, 1, 3])]}
    res, info, log = GF.run_graphs([g], str(tmp_path))
    assert res[0] is not None, (info, log[-2000:])
    assert np.array_equal(res[0], oracle.run_graph(g))


@pytest.mark.gpu
def test_layout_inference_on_a_channel_fastest_network(tmp_path, oracle):
    """What an NHWC front end hands over (src/tim/transform/layout_inference.cc): CWHN uint8
    activations, IcWHOc kernels. conv3x3+relu6 -> depthwise3x3 -> 1x1 conv -> residual Add ->
    avg pool -> Reshape -> FullyConnected -> Softmax. The rewritten graph must give what the
    oracle computes operator by operator with explicit transposes around every CWHN operator;
    at debug log level the plan shows one permute behind the input and one in front of Reshape."""
    rng = np.random.default_rng(21)
    c0, c1, w, h, n, classes = 8, 16, 12, 10, 2, 10
    q, T, OP = GF.asym, GF.tensor, GF.op
    u8 = lambda *s: rng.integers(0, 256, int(np.prod(s)), dtype=np.uint8)
    cw = dict(layout="CWHN", kernel_layout="IcWHOc", pad_type="AUTO")
    g = {"test": "nhwc_net", "output": 18, "layout_inference": True, "tensors": [
        T(0, "UINT8", "INPUT", [c0, w, h, n], q(0.5, 128), u8(c0, w, h, n)),
        T(1, "UINT8", "CONSTANT", [c0, 3, 3, c1], q(0.02, 120), u8(c0, 3, 3, c1)),
        T(2, "INT32", "CONSTANT", [c1], q(0.01, 0), rng.integers(-500, 500, c1, dtype=np.int32)),
        T(3, "UINT8", "TRANSIENT", [c1, w, h, n], q(4.0, 128)),
        T(4, "UINT8", "CONSTANT", [c1, 3, 3, 1], q(0.03, 130), u8(c1, 3, 3, 1)),
        T(5, "INT32", "CONSTANT", [c1], q(0.12, 0), rng.integers(-500, 500, c1, dtype=np.int32)),
        T(6, "UINT8", "TRANSIENT", [c1, w, h, n], q(16.0, 110)),
        T(7, "UINT8", "CONSTANT", [c1, 1, 1, c1], q(0.02, 125), u8(c1, 1, 1, c1)),
        T(8, "INT32", "CONSTANT", [c1], q(0.32, 0), rng.integers(-500, 500, c1, dtype=np.int32)),
        T(9, "UINT8", "TRANSIENT", [c1, w, h, n], q(60.0, 120)),
        T(10, "UINT8", "TRANSIENT", [c1, w, h, n], q(64.0, 100)),
        T(11, "UINT8", "TRANSIENT", [c1, w // 2, h // 2, n], q(64.0, 100)),
        T(12, "UINT8", "TRANSIENT", [c1 * (w // 2) * (h // 2), n], q(64.0, 100)),
        T(13, "UINT8", "CONSTANT", [c1 * (w // 2) * (h // 2), classes], q(1e-5, 128), u8(c1 * (w // 2) * (h // 2), classes)),
        T(14, "INT32", "CONSTANT", [classes], q(0.00064, 0), rng.integers(-2000, 2000, classes, dtype=np.int32)),
        T(15, "UINT8", "TRANSIENT", [classes, n], q(0.5, 128)),
        T(18, "FLOAT32", "OUTPUT", [classes, n])],
        "ops": [OP("CONV2D", [0, 1, 2], [3], pad=[1, 1, 1, 1], ksize=[3, 3], weights=c1, **cw),
                OP("CONV2D", [3, 4, 5], [6], pad=[1, 1, 1, 1], ksize=[3, 3], weights=c1, multiplier=1, **cw),
                OP("CONV2D", [6, 7, 8], [9], pad=[0, 0, 0, 0], ksize=[1, 1], weights=c1, **cw),
                OP("ADD", [9, 3], [10]),
                OP("POOL", [10], [11], pool_type="AVG", ksize=[2, 2], stride=[2, 2], pad=[0, 0, 0, 0], layout="CWHN", pad_type="AUTO"),
                OP("RESHAPE", [11], [12], new_shape=[c1 * (w // 2) * (h // 2), n]),
                OP("FCL", [12, 13, 14], [15], axis=0, weights=classes),
                OP("SOFTMAX", [15], [18], beta=0.05, sm_axis=0)]}
    # applications declare TRANSIENT tensors without a shape (samples/lenet/lenet_asymu8.cc:127-160): the
    # graph goes to the runtime that way, the oracle gets the shapes spelled out
    bare = copy.deepcopy(g)
    for t in bare["tensors"]:
        if t["attr"] == "TRANSIENT":
            t["shape"] = []
    res, info, log = GF.run_graphs([bare], str(tmp_path), env={"VSI_NN_LOG_LEVEL": "3"})
    assert res[0] is not None, (info, log[-3000:])
    want = oracle.run_graph(g)
    assert np.allclose(res[0], want, rtol=0, atol=1e-6), (res[0][:10], want[:10])
    logits = copy.deepcopy(g)        # the uint8 logits bit for bit
    logits["test"] = "nhwc_net_logits"
    logits["ops"] = logits["ops"][:-1]
    logits["tensors"] = logits["tensors"][:-1]
    logits["tensors"][-1]["attr"] = "OUTPUT"
    logits["output"] = 15
    res2, info2, log2 = GF.run_graphs([logits], str(tmp_path), env={"VSI_NN_LOG_LEVEL": "3"})
    assert res2[0] is not None, (info2, log2[-3000:])
    assert np.array_equal(res2[0], oracle.run_graph(logits))
    plan = [l for l in log2.splitlines() if "uid" in l and "->" in l]
    assert sum("transpose" in l for l in plan) == 2, plan


@pytest.mark.gpu
@pytest.mark.parametrize("handles", [False, True, "platform"], ids=["copies", "io_handles", "platform"])
def test_repeated_runs_follow_the_inputs(tmp_path, oracle, handles):
    """Run() may be called again and again with the inputs re-filled in between
    (src/tim/vx/graph.cc:378-391): six runs with the input alternating between two images,
    host copies and synchronisations in between as an application would have them; every
    run must equal the oracle's result for the image it was given. With io_handles the graph's
    input and output are Graph::CreateIOTensor tensors on buffers of the caller: filled in place
    and handed over with FlushCacheForHandle, read in place after InvalidateCacheForHandle, and
    every re-run brings a new input buffer in through SwapHandle (the old one, overwritten, must
    not be read again) - the delegate's zero-copy protocol (include/tim/vx/tensor.h:154-166)."""
    w, x = _lenet_data()
    rng = np.random.default_rng(11)
    other = rng.integers(0, 256, x.size, dtype=np.uint8)
    g = GRAPHS.lenet_asymu8(w, x)
    logits = copy.deepcopy(g)
    logits["test"] = "lenet_logits_replay"
    logits["ops"] = logits["ops"][:-1]
    logits["tensors"] = logits["tensors"][:-1]
    logits["tensors"][15]["attr"] = "OUTPUT"
    logits["output"] = 15
    in_id = next(t["id"] for t in logits["tensors"] if t["attr"] == "INPUT")
    logits["reruns"] = [{in_id: other}, {in_id: x}, {in_id: other}, {in_id: other}, {in_id: x}]
    logits["handles"] = handles is True
    logits["platform"] = handles == "platform"   # re-submitted and triggered per run
    want_x = oracle.run_graph(logits)
    alt = copy.deepcopy(logits)
    {t["id"]: t for t in alt["tensors"]}[in_id]["data"] = other
    want_other = oracle.run_graph(alt)
    assert not np.array_equal(want_x, want_other)
    expect = [want_x, want_other, want_x, want_other, want_other, want_x]
    res, info, log = GF.run_graphs([logits], str(tmp_path))
    runs = [res[0]] + info["lenet_logits_replay"]["reruns"]
    assert len(runs) == 6 and all(r is not None for r in runs), (info, log[-2000:])
    for i, (got, want) in enumerate(zip(runs, expect)):
        assert np.array_equal(got, want), i


@pytest.mark.gpu
@pytest.mark.parametrize("batch,res", [(2, 224), (3, 96)])
def test_mobilenet_v2_graph_bit_exact(tmp_path, oracle, batch, res):
    g = GRAPHS.mobilenet_v2(batch=batch, res=res, seed=batch)
    out, info, log = GF.run_graphs([g], str(tmp_path), env={"VSI_NN_LOG_LEVEL": "3"})
    assert out[0] is not None, (info, log[-2000:])
    ref = oracle.run_graph(g)
    assert len(np.unique(ref)) > 30  # the synthetic network is not degenerate
    assert np.array_equal(out[0], ref), int((out[0] != ref).sum())
    # the ten residual Adds ride on the projection convolutions in front of them: no Add kernel in the plan
    plan = [l for l in log.splitlines() if "uid" in l and "->" in l]
    assert sum("pwconv_add_i8" in l or "pwconv_reg_add_i8" in l or "pwconv_add_blocked_i8" in l for l in plan) == 10 and not any("ADD" in l for l in plan), plan


@pytest.mark.gpu
@pytest.mark.parametrize("side,batch", [(7, 3), (5, 1), (8, 2)])
def test_blocked_plan_with_a_copy_in(tmp_path, oracle, side, batch):
    """A run of small-plane convolutions behind an INPUT tensor: the executor keeps its TRANSIENT tensors channel-blocked;
    the input - read by the expansion and, as the residual, by the Add - is copied into that order once; the average
    pooling leaves the plan. Bit for bit the WHCN plan's result."""
    g = GRAPHS._Builder(side * 10 + batch)
    x = g.new("UINT8", "INPUT", [side, side, 64, batch], GF.asym(0.05, 128),
              g.rng.integers(0, 256, size=side * side * 64 * batch, dtype=np.uint8))
    x["_rms"] = 74.0
    h = g.conv(x, 192, 1, 1, "RELU6")
    h = g.conv(h, 192, 3, 1, "RELU6", depthwise=True)
    h = g.conv(h, 64, 1, 1, None)
    h = g.add(x, h)
    h = g.conv(h, 96, 1, 1, "RELU6")
    out = g.new("UINT8", "OUTPUT", [1, 1, 96, batch], h["quant"])
    g.ops.append(GF.op("POOL", [h["id"]], [out["id"]], pad_type="VALID", pool_type="AVG", ksize=[side, side], stride=[side, side]))
    graph = {"test": "blocked_copy_in_%d_%d" % (side, batch), "tensors": g.tensors, "ops": g.ops, "output": out["id"]}
    want = oracle.run_graph(graph)
    assert len(np.unique(want)) > 8
    got, info, log = GF.run_graphs([graph], str(tmp_path / "blocked"), env={"VSI_NN_LOG_LEVEL": "3"})
    assert got[0] is not None, (info, log[-2000:])
    assert np.array_equal(got[0], want), int((got[0] != want).sum())
    plan = [l for l in log.splitlines() if "uid" in l and "->" in l]
    assert sum("layout_to_blocked" in l for l in plan) == 1 and sum("_blocked_i8" in l for l in plan) == 5, plan
    assert sum("pwconv_add_blocked_i8" in l for l in plan) == 1 and not any("ADD" in l for l in plan), plan
    plain, info, log = GF.run_graphs([graph], str(tmp_path / "whcn"), env={"VSI_NN_LOG_LEVEL": "3", "TVX_BLOCKED_LAYOUT": "0"})
    assert np.array_equal(plain[0], want) and "blocked" not in log


def _pool_graph(name, in_shape, out_shape, pool_type, form, ksize, stride, dt="UINT8", in_q=(0.5, 12), out_q=(0.5, 12)):
    rng = np.random.default_rng(len(name))
    lo, hi = (0, 256) if dt == "UINT8" else (-128, 128)
    x = rng.integers(lo, hi, int(np.prod(in_shape))).astype(np.uint8 if dt == "UINT8" else np.int8)
    ts = [GF.tensor(0, dt, "INPUT", in_shape, GF.asym(*in_q), x),
          GF.tensor(1, dt, "OUTPUT", out_shape, GF.asym(*out_q))]
    ops = [GF.op("POOL", [0], [1], pool_type=pool_type, pool_1d=form, ksize=ksize, stride=stride)]
    return {"test": name, "tensors": ts, "ops": ops, "output": 1}


@pytest.mark.gpu
def test_pool2d_global_and_adaptive_constructors(tmp_path, oracle):
    """Pool2d's two constructors that take sizes instead of a window (include/tim/vx/ops/pool2d.h:87-99,
    src/tim/vx/ops/pool2d.cc:62-93): global pooling (window = stride = input size) and adaptive pooling
    (stride = floor(in / out), window = in - (out - 1) * stride). The runner calls the constructors; the
    expectation is the oracle's pooling over the window those rules give, written out here."""
    cases, wants = [], []
    for pool_type in ("MAX", "AVG"):
        g = _pool_graph("global_" + pool_type, [7, 5, 24, 3], [1, 1, 24, 3], pool_type, "global", [7, 5], [7, 5],
                        out_q=(0.75, 3))
        cases.append(g)
        e = copy.deepcopy(g)
        e["ops"][0]["attrs"].update(pool_1d=False, ksize=[7, 5], stride=[7, 5])
        wants.append(oracle.run_graph(e))
        for (iw, ih), (ow, oh) in (((12, 10), (4, 3)), ((9, 9), (2, 2)), ((16, 8), (16, 8))):
            g = _pool_graph("adaptive_%s_%dx%d_to_%dx%d" % (pool_type, iw, ih, ow, oh), [iw, ih, 8, 2], [ow, oh, 8, 2],
                            pool_type, "adaptive", [iw, ih], [ow, oh], dt="INT8", in_q=(0.1, -4), out_q=(0.13, 2))
            cases.append(g)
            sw, sh = iw // ow, ih // oh
            e = copy.deepcopy(g)
            e["ops"][0]["attrs"].update(pool_1d=False, ksize=[iw - (ow - 1) * sw, ih - (oh - 1) * sh], stride=[sw, sh])
            wants.append(oracle.run_graph(e))
    res, info, log = GF.run_graphs(cases, str(tmp_path))
    for c, got, want in zip(cases, res, wants):
        assert got is not None, (c["test"], info.get(c["test"]), log[-1500:])
        assert np.array_equal(got, want), c["test"]
    assert all(len(np.unique(w)) > 4 for w in wants)


@pytest.mark.gpu
def test_operators_arrive_through_clone(tmp_path, oracle):
    """Operation::Clone (include/tim/vx/operation.h:46): every operator of the sample network and of a graph
    with the sized Pool2d constructors is created in a second graph and cloned into the one that runs; the
    clone must carry every attribute (pads, strides, multiplier, weights, axis, the pooling window)."""
    w, x = _lenet_data()
    g = GRAPHS.lenet_asymu8(w, x)
    g["test"] = "lenet_cloned"
    g["clone"] = True
    p = _pool_graph("adaptive_cloned", [12, 10, 8, 2], [4, 3, 8, 2], "AVG", "adaptive", [12, 10], [4, 3])
    p["clone"] = True
    e = copy.deepcopy(p)
    e["ops"][0]["attrs"].update(pool_1d=False, ksize=[12 - 3 * 3, 10 - 2 * 3], stride=[3, 3])
    m = GRAPHS.mobilenet_v2(batch=1, res=32)
    m["test"] = "mobilenet_cloned"
    m["clone"] = True
    res, info, log = GF.run_graphs([g, p, m], str(tmp_path))
    assert all(r is not None for r in res), (info, log[-1500:])
    assert np.array_equal(res[0], oracle.run_graph(g))
    assert np.array_equal(res[1], oracle.run_graph(e))
    assert np.array_equal(res[2], oracle.run_graph(m))


def test_compile_option_carries_the_device(tmp_path):
    """CompileOption::setDeviceId / getDeviceId (include/tim/vx/compile_option.h:45-48; the graph hands the
    index to the driver at src/tim/vx/graph.cc:345-348): a graph created for a GPU the machine does not have
    must not compile; index 0 is the GPU this runtime drives."""
    g = _pool_graph("device_7", [4, 4, 8, 1], [2, 2, 8, 1], "MAX", False, [2, 2], [2, 2])
    g["device"] = 7
    ok = _pool_graph("device_0", [4, 4, 8, 1], [2, 2, 8, 1], "MAX", False, [2, 2], [2, 2])
    ok["device"] = 0
    res, info, log = GF.run_graphs([g, ok], str(tmp_path))
    assert res[0] is None and info["device_7"]["fail"] == "compile"
    if _has_gpu():
        assert "compiled for device 7" in log
        assert res[1] is not None
