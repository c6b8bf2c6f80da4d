"""Float16 1x1 convolutions with their pixels in registers: ends of pixel groups, images, channel steps and output tiles, both ways of sharing a
reduction, against the oracle and, where infinities are among the inputs, against each product by itself."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu

# batch, channels, height, width, output channels
LAYERS = [(1, 1, 2, 4, 1), (3, 8, 3, 3, 17), (2, 31, 5, 5, 16), (1, 32, 16, 8, 33), (5, 33, 7, 9, 40), (2, 64, 11, 13, 15), (1, 97, 9, 31, 65), (2, 128, 12, 12, 48),
          (3, 40, 1, 41, 130), (2, 129, 6, 7, 20), (1, 200, 8, 8, 96), (2, 260, 5, 7, 31), (1, 515, 4, 5, 64), (2, 777, 3, 4, 18), (1, 1024, 3, 3, 16)]


def _exact(x, wt, b, act):
    """The convolution in 64 bits; by how much a result may be off: c + 1 additions of float32, each by at most a unit of its last place of what the
    magnitudes add up to, and half a unit of float16's last place; and the convolution without its last channel."""
    x, wt, b = x.astype(np.float64), wt.astype(np.float64), b.astype(np.float64)[:, None]
    c = wt.shape[1]

    def activated(v):
        return v if act == 0 else np.clip(v, 0, None if act == 1 else 6)
    exact, lost = wt @ x + b, wt[:, :-1] @ x[:, :-1] + b
    bound = (c + 1) * 2.0 ** -23 * (np.abs(wt) @ np.abs(x) + np.abs(b))
    return activated(exact), bound + 2.0 ** -11 * (np.abs(exact) + bound) + 2.0 ** -25, activated(lost)


@pytest.mark.parametrize("act", [0, 1, 2])
@pytest.mark.parametrize("ks", [1, 4])
@pytest.mark.parametrize("layer", LAYERS)
def test_pointwise_f16_in_registers(oracle, layer, ks, act, monkeypatch):
    n, c, h, w, oc = layer
    if ks == 1 and c > 128:
        pytest.skip("a wavefront holds 128 channels")
    rng = np.random.default_rng(8800 + c + oc)
    x, wt, b, kws = conv_case(rng, mult=0, mode="f16", n=n, c=c, h=h, w=w, oc=oc, kh=1, kw=1, stride=[1, 1], dil=[1, 1], pad=[0] * 4)
    monkeypatch.setenv("TVX_PWCONV_F16", str(ks))
    want = oracle.conv2d(x, wt, b, act=act, **kws).astype(np.float64).reshape(n, oc, h * w)
    exact, bound, lost = _exact(x.reshape(n, c, h * w), wt.reshape(oc, c), b, act)
    assert (np.abs(want - exact) <= bound).all()
    for waves in (1, 1 << 20):   # all output tiles after one another, each by itself
        monkeypatch.setenv("TVX_PWCONV_F16_WAVES", str(waves))
        got = TC.gpu_conv2d(x, wt, b, act=act, want_kernel="pwconv_reg_f16", **kws).astype(np.float64).reshape(n, oc, h * w)
        assert (np.abs(got - exact) <= bound).all(), np.max(np.abs(got - exact) / bound)
        assert c == 1 or act or (np.abs(got - lost) > bound).mean() > 0.5   # (the bound tells the sum from one without its last channel)


@pytest.mark.parametrize("ks,c", [(1, 13), (1, 100), (4, 133)])
def test_an_infinity_stays_with_its_pixel(ks, c, monkeypatch):
    n, h, w, oc = 2, 5, 7, 20
    rng = np.random.default_rng(8900 + c)
    x, wt, b, kws = conv_case(rng, mult=0, mode="f16", n=n, c=c, h=h, w=w, oc=oc, kh=1, kw=1, stride=[1, 1], dil=[1, 1], pad=[0] * 4)
    wt = np.abs(wt) + np.float16(0.125)
    x = np.clip(x, -4, 4)
    x.reshape(n, c, h * w)[1, c - 1, 3] = np.inf
    x.reshape(n, c, h * w)[0, 0, h * w - 1] = -np.inf
    monkeypatch.setenv("TVX_PWCONV_F16", str(ks))
    got = TC.gpu_conv2d(x, wt, b, act=0, want_kernel="pwconv_reg_f16", **kws).reshape(n, oc, h * w)
    odd = np.zeros((n, h * w), bool)
    odd[1, 3] = odd[0, -1] = True
    assert (got[1, :, 3] == np.inf).all() and (got[0, :, -1] == -np.inf).all()
    assert np.isfinite(got.transpose(0, 2, 1)[~odd]).all()


@pytest.mark.parametrize("n,c,h,w,oc,mine", [
    (1, 64, 1, 577, 17, True), (1, 64, 24, 24, 17, True), (4, 64, 16, 16, 16, True), (4, 65, 16, 16, 16, True), (3, 64, 15, 17, 16, True), (4, 64, 16, 16, 17, True),
    (2, 300, 31, 37, 40, True), (1, 1025, 25, 25, 20, False), (1, 40, 512, 256, 50, True), (1, 40, 512, 257, 50, True), (1, 70, 363, 362, 49, True),
    # a group of eight pixels, one less; a single result of a handful of pixels and of many; 1024 channels of few
    (1, 24, 2, 4, 9, True), (9, 24, 1, 7, 9, False), (5, 16, 3, 3, 1, True), (2, 64, 120, 128, 6, True), (3, 1024, 4, 4, 24, True)])
@pytest.mark.parametrize("levers", [{}, {"TVX_CONV_TILE": "0"}, {"TVX_CONV_TILE": "1"}, {"TVX_NO_CONV_IGEMM_F16": "1", "TVX_NO_CONV_GEMM": "1"}])
def test_which_layers(oracle, n, c, h, w, oc, mine, levers, monkeypatch):
    """Planes of eight pixels and more, up to 1024 channels; the levers of the kernels asked behind it are theirs alone."""
    for k, v in levers.items():
        monkeypatch.setenv(k, v)
    x, wt, b, kws = conv_case(np.random.default_rng(8990), mult=0, mode="f16", n=n, c=c, h=h, w=w, oc=oc, kh=1, kw=1, stride=[1, 1], dil=[1, 1], pad=[0] * 4)
    want = oracle.conv2d(x, wt, b, act=1, **kws)
    got = TC.gpu_conv2d(x, wt, b, act=1, want_kernel="pwconv_reg_f16" if mine else ("conv2d_tile_f16", "conv2d_gemm_f16", "conv2d_igemm_f16", "conv2d_generic"), **kws)
    assert np.allclose(got.astype(np.float32), want.astype(np.float32), rtol=5e-3, atol=2e-2)
