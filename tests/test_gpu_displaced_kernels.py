"""Kernels whose layers newer ones mostly take, on the layers that are still theirs and, by the newer ones' levers, on their old ones; and
which kernel takes a layer of its own accord. Exact against the oracle."""
import numpy as np
import pytest

import test_gpu_fused_small_nets as SN
import test_gpu_parity as PT
import tvx_case as TC
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu

IGEMM_POOL = [c for c in SN.CONV_POOL if c["kernel"] == "conv2d_igemm_maxpool_i8"]
# an image too large for LDS; rows of fewer than four columns
OWN_POOL = [dict(n=2, c=64, h=40, w=40, oc=24, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1], kernel="conv2d_igemm_maxpool_i8"),
            dict(n=1, c=40, h=10, w=2, oc=20, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1], kernel="conv2d_igemm_maxpool_i8")]


@pytest.mark.parametrize("tile", [0, 32])
@pytest.mark.parametrize("mode", ["u8", "i8pc"])
@pytest.mark.parametrize("gi", range(len(IGEMM_POOL) + len(OWN_POOL)))
def test_pooled_implicit_gemm(oracle, gi, mode, tile, monkeypatch):
    if gi < len(IGEMM_POOL):
        monkeypatch.setenv("TVX_CONV_POOL", "0")
    else:
        case = SN.conv_case

        def fitted(*args, **kws):  # (the largest of four sums of 576 products would mostly lie on the clamp)
            x, w, b, kws = case(*args, **kws)
            kws["in_q"] = (kws["in_q"][0] / 8, kws["in_q"][1])
            return x, w, b, kws
        monkeypatch.setattr(SN, "conv_case", fitted)
    monkeypatch.setattr(SN, "CONV_POOL", IGEMM_POOL + OWN_POOL)
    TC.expect_variant(monkeypatch, "conv2d_igemm_maxpool_i8")
    SN.test_conv2d_with_fused_max_pool(oracle, gi, mode, tile, monkeypatch)


@pytest.mark.parametrize("mode", ["u8", "i8pc", "u8pc"])
@pytest.mark.parametrize("gi", range(len(PT.DWP_GRID)))
def test_depthwise_planes(oracle, gi, mode, monkeypatch):
    n, c, h, w, kh, kw, stride, dil, pad = PT.DWP_GRID[gi]
    monkeypatch.setenv("TVX_DWCONV_REG", "0")
    dwords = kh == kw == 3 and stride[0] == stride[1] and dil == [1, 1]
    TC.expect_variant(monkeypatch, "dwconv_rows_i8" if dwords else "dwconv_planes_i8")
    PT.test_depthwise_planes_shapes(oracle, gi, mode)


@pytest.mark.parametrize("c,h,w,stride,kernel", [
    (4, 9, 132, 1, "dwconv_reg_i8"), (3, 9, 52, 1, "dwconv3x3_i8"),      # outputs of a row in 33 of 64 lanes, in 13 of 16
    (3, 9, 136, 1, "dwconv3x3_i8"), (2, 9, 264, 1, "dwconv_reg_i8"),     # rows of whole 8-byte units; rows over 256 columns
    (5, 14, 14, 1, "dwconv_reg_i8"), (5, 7, 7, 1, "dwconv_reg_i8"),      # no whole dwords
    (3, 20, 24, 2, "dwconv3x3_i8"), (3, 20, 27, 2, "dwconv_reg_i8")])
def test_which_kernel_takes_a_quantized_3x3_layer(oracle, c, h, w, stride, kernel):
    pad = [1, 1, 1, 1] if stride == 1 else [0, 1, 0, 1]
    rng = np.random.default_rng(7400 + w)
    for mode in ("u8", "i8pc"):
        x, wt, b, kws = conv_case(rng, n=2, c=c, h=h, w=w, oc=0, kh=3, kw=3, stride=[stride, stride], dil=[1, 1], pad=pad, mult=1, mode=mode)
        got = TC.gpu_conv2d(x, wt, b, act=2, want_variant=kernel, **kws)
        assert np.array_equal(got, oracle.conv2d(x, wt, b, act=2, **kws))


@pytest.mark.parametrize("room,kernel", [(9 * 128 * 128, "dwconv3x3_i8"), (9 * 128 * 128 - 1, "dwconv_rows_i8")])
@pytest.mark.parametrize("sign", [1, -1])
def test_depthwise_biases_at_the_ends_of_their_range(oracle, sign, room, kernel):
    """The sums of the register stencil saturate: a bias that leaves them no room goes to the kernel whose sums wrap around."""
    n, c, h, w = 2, 6, 16, 16
    rng = np.random.default_rng(7600)
    x, wt = rng.integers(-128, 128, n * c * h * w).astype(np.int8), rng.integers(-128, 128, c * 9).astype(np.int8)
    b = rng.integers(-4096, 4097, c).astype(np.int32)
    b[1] = sign * (2 ** 31 - 1 - room)
    scales = np.full(c, 0.02, np.float32)
    kws = dict(in_shape=[w, h, c, n], w_shape=[3, 3, 1, c], out_shape=[w, h, c, n], stride=[1, 1], dilation=[1, 1], pad_left=1, pad_top=1, multiplier=1,
               in_dtype=1, w_dtype=1, out_dtype=1, in_q=(0.05, 0), w_q=(1.0, 0, scales), out_q=(0.6, 3))
    want = oracle.conv2d(x, wt, b, act=0, **kws)
    assert (want.reshape(n, c, -1)[:, 1] == (127 if sign > 0 else -128)).all() and len(np.unique(want)) > 100
    got = TC.gpu_conv2d(x, wt, b, act=0, want_variant=kernel, **kws)
    assert np.array_equal(got, want), int((got != want).sum())


@pytest.mark.parametrize("dtype,w,h", [(0, 40, 70), (1, 61, 46), (2, 60, 76), (3, 42, 42)])
def test_averages_of_many_planes_by_wavefronts(oracle, dtype, w, h):
    """Up to eight planes a compute unit, a workgroup each; of more, planes just below their type's line take a wavefront, those beyond a workgroup."""
    import torch
    planes, base = 8 * torch.cuda.get_device_properties(0).multi_processor_count, {0: "avgpool_plane_i8", 1: "avgpool_plane_i8", 2: "pool2d_generic", 3: "pool2d_generic"}[dtype]
    rng = np.random.default_rng(7500 + dtype)
    T, p = TC.tvx(), TC.tvx().Pool2dDesc()
    seen = []
    for n, cols in ((planes - 1, w), (planes, w), (planes, w + 2)):
        p.in_w, p.in_h, p.channels, p.batch, p.out_w, p.out_h, p.k_w, p.k_h, p.stride_w, p.stride_h = cols, h, n, 1, 1, 1, cols, h, 1, 1
        p.pool_type, p.dtype, p.in_scale, p.out_scale = T.POOL_AVG, dtype, 0.5, 0.5
        op = T.pool2d_create(p)
        seen.append(op.variant)
        x = rng.integers(0, 100, n * cols * h).astype(TC.NP_OF[dtype])
        y = TC.device_out(n, TC.NP_OF[dtype])
        op.run(TC.to_device(x), None, y)
        got, want = y.cpu().numpy().astype(np.float64), x.astype(np.float64).reshape(n, -1).mean(1)
        # (whole codes, ties to even; float32 sums of under 5000 values to 2^-19 of them, then a rounding to float16: 2^-11)
        assert np.array_equal(got, np.rint(want)) if dtype < 2 else np.abs(got / want - 1).max() <= (2.0 ** -10 if dtype == 2 else 2.0 ** -18)
        op.close()
    assert seen == ["pool2d_plane_sum", base, "pool2d_plane_sum"]


def test_launches_of_no_more_threads_than_there_can_be():
    """2^32 threads: kernels that take more of them than the ones before decline from there on. (Nothing runs: these tensors have gigabytes.)"""
    T = TC.tvx()
    p = T.Pool2dDesc()
    p.in_w, p.in_h, p.channels, p.out_w, p.out_h, p.k_w, p.k_h, p.stride_w, p.stride_h = 64, 256, 64, 1, 1, 64, 256, 1, 1
    p.pool_type = T.POOL_AVG
    for dtype, kernel in ((T.U8, "avgpool_plane_i8"), (T.F16, "pool2d_generic"), (T.F32, "pool2d_generic")):
        p.dtype, p.in_scale, p.out_scale = dtype, 0.5, 0.5
        for p.batch, want in ((2 ** 18 - 1, "pool2d_plane_sum"), (2 ** 18, kernel)):
            op = T.pool2d_create(p)
            assert op.variant == want, (dtype, p.batch, op.variant)
            op.close()
    rng = np.random.default_rng(5)
    x, w, b, kws = conv_case(rng, n=1, c=17, h=8, w=8, oc=128, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1], mult=0, mode="u8")
    for n, want in ((2 ** 22 - 1, "conv2d_pool_i8"), (2 ** 22, "conv2d_igemm_maxpool_i8")):
        kws["in_shape"][3] = kws["out_shape"][3] = n
        op = T.conv2d_pool_create(*SN._descs(T, kws, 0, []), w, b)
        assert op.variant == want, (n, op.variant)
        op.close()
