"""Short-window convolutions gathered into registers (kernels three and five taps wide): runs of one, two and five tiles a wavefront,
every number of reduction steps, dilated rows, padding as wide as a window reaches, planes and pooled planes that end inside a tile, strides,
weight zero points at the ends of their range, and outputs of both types. Exact against the oracle."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu

CASES = [
    dict(n=3, c=1, h=9, w=7, oc=5, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1]),
    dict(n=2, c=7, h=11, w=13, oc=33, kh=3, kw=3, stride=[2, 1], dil=[1, 1], pad=[0, 2, 2, 0]),      # 21 kernel rows: three steps
    dict(n=2, c=4, h=12, w=10, oc=70, kh=3, kw=3, stride=[1, 2], dil=[1, 2], pad=[1, 1, 3, 0]),      # dilated rows, two steps
    dict(n=1, c=2, h=16, w=16, oc=24, kh=5, kw=5, stride=[1, 1], dil=[1, 1], pad=[4, 4, 4, 4]),      # two steps of five taps
    dict(n=2, c=1, h=5, w=5, oc=32, kh=5, kw=5, stride=[1, 1], dil=[1, 1], pad=[4, 4, 4, 4]),        # a single tap inside the image
    dict(n=4, c=3, h=33, w=35, oc=32, kh=1, kw=3, stride=[2, 2], dil=[1, 1], pad=[1, 1, 0, 0]),
    dict(n=1, c=1, h=1, w=8, oc=1, kh=1, kw=5, stride=[1, 1], dil=[1, 1], pad=[2, 2, 0, 0]),         # the smallest tensor a run is read from
]


@pytest.mark.parametrize("run", [1, 2, 5])
@pytest.mark.parametrize("mode", ["u8", "i8pc", "u8zp0"])
@pytest.mark.parametrize("ci", range(len(CASES)))
def test_register_gather(oracle, monkeypatch, ci, mode, run):
    monkeypatch.setenv("TVX_IM2COL_RUN", str(run))
    rng = np.random.default_rng(8700 + ci)
    x, w, b, kws = conv_case(rng, mult=0, mode="u8" if mode == "u8zp0" else mode, **CASES[ci])
    if mode == "u8zp0":  # (every weight counts 120-odd more: a wider output scale)
        kws["w_q"] = (kws["w_q"][0], 0, None)
        kws["out_q"] = (kws["out_q"][0] * 2, kws["out_q"][1])
    want = oracle.conv2d(x, w, b, act=2, **kws)
    got = TC.gpu_conv2d(x, w, b, act=2, want_kernel="conv2d_im2col_i8", want_variant="conv2d_im2col_reg_i8", **kws)
    assert np.array_equal(got, want), (int((got != want).sum()), np.flatnonzero(got != want)[:8])


@pytest.mark.parametrize("pool", [False, True])
@pytest.mark.parametrize("in_zp", [-128, 127])
def test_biases_at_the_ends_of_their_range(oracle, in_zp, pool):
    """Accumulators within 32 bits whose bias, with the zero points' constants folded in, is not: the sums wrap around and back."""
    rng = np.random.default_rng(8750)
    n, c, k, oc, side = 2, 3, 3, 40, 10
    x = (in_zp + (1 if in_zp < 0 else -1) * rng.integers(0, 9, n * c * (side + 2) ** 2)).astype(np.int8)
    w = rng.integers(100, 128, oc * c * k * k).astype(np.int8)
    room = 9 * c * k * k * 128                       # what a window adds to the bias or takes from it
    folded = c * k * k * 128 * 100                   # what the input zero point does at least
    sign = 1 if in_zp < 0 else -1
    b = rng.integers(-4096, 4097, oc)
    b[::2] = sign * (2 ** 31 - 1 - rng.integers(room, folded // 2, oc)[::2])
    scales = np.exp(rng.uniform(np.log(0.002), np.log(0.05), oc)).astype(np.float32)
    kws = dict(in_shape=[side + 2, side + 2, c, n], w_shape=[k, k, c, oc], out_shape=[side, side, oc, n], stride=[1, 1], dilation=[1, 1], pad_left=0,
               pad_top=0, multiplier=0, in_dtype=1, w_dtype=1, out_dtype=1, in_q=(0.05, in_zp), w_q=(1.0, 0, scales), out_q=(0.3, -3))
    want = oracle.conv2d(x, w, b.astype(np.int32), act=0, **kws)
    assert (want.reshape(n, oc, -1)[:, ::2] == (127 if sign > 0 else -128)).all() and len(np.unique(want)) > 50
    if not pool:
        got = TC.gpu_conv2d(x, w, b.astype(np.int32), act=0, want_variant="conv2d_im2col_reg_i8", **kws)
        assert np.array_equal(got, want), int((got != want).sum())
        return
    import torch
    import test_gpu_fused_small_nets as SN
    want = want.reshape(n * oc, side // 2, 2, side // 2, 2).max(axis=(2, 4)).reshape(-1)
    keep = []
    op = TC.tvx().conv2d_pool_create(*SN._descs(TC.tvx(), kws, 0, keep), w, b.astype(np.int32))
    assert op.variant == "conv2d_im2col_reg_maxpool_i8"
    xd, yd = TC.to_device(x), TC.device_out(want.size, np.int8)
    op.run(xd, None, yd)
    torch.cuda.synchronize()
    got = yd.cpu().numpy()
    op.close()
    assert np.array_equal(got, want), int((got != want).sum())
