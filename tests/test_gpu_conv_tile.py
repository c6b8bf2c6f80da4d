"""The one-tile-per-workgroup convolution (dense and grouped; int8, float16, float32) at the edges of its tiles: every way
its wavefronts share a tile, on planes that end inside tiles, granules, column groups and channel blocks."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu

SHAPES = range(8)   # 256 x 64 down to 32 x 32 (pixels x channels)
KERNEL = {"u8": "conv2d_tile_i8", "i8pc": "conv2d_tile_i8", "f16": "conv2d_tile_f16", "f32": "conv2d_tile_f32"}

CASES = {
    # one 16-byte granule with three channels, an odd number of reduction steps, rows of one more than whole column groups
    "shallow": dict(n=2, c=3, h=11, w=17, oc=33, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1]),
    # several images per tile, a batch that does not fill the last one, planes narrower than a column group
    "images": dict(n=5, c=20, h=7, w=5, oc=40, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1]),
    # stride 2, uneven pads, output rows that are no multiple of four
    "strided": dict(n=1, c=40, h=23, w=30, oc=65, kh=5, kw=3, stride=[2, 2], dil=[1, 1], pad=[0, 1, 2, 1]),
    "dilated": dict(n=2, c=16, h=14, w=19, oc=24, kh=3, kw=3, stride=[1, 1], dil=[2, 3], pad=[3, 3, 2, 2]),
    "grouped": dict(n=3, c=36, h=9, w=13, oc=20, kh=3, kw=3, stride=[1, 2], dil=[1, 1], pad=[1, 1, 1, 1], groups=4),
    # 1 x 1: the image as one row (its last pixels are read from in front), and under a stride
    "pointwise": dict(n=3, c=24, h=5, w=29, oc=70, kh=1, kw=1, stride=[1, 1], dil=[1, 1], pad=[0, 0, 0, 0]),
    "pointwise_strided": dict(n=2, c=50, h=15, w=13, oc=32, kh=1, kw=1, stride=[2, 2], dil=[1, 1], pad=[0, 0, 0, 0]),
    # a window wider than the image, nearly all padding
    "window": dict(n=2, c=17, h=4, w=3, oc=16, kh=7, kw=7, stride=[1, 1], dil=[1, 1], pad=[3, 3, 3, 3]),
    # more channels than a tile's window fits LDS with: several chunks, the last one with an empty granule
    "chunks": dict(n=1, c=300, h=20, w=21, oc=33, kh=5, kw=5, stride=[1, 1], dil=[1, 1], pad=[2, 2, 2, 2]),
    "row": dict(n=2, c=12, h=1, w=61, oc=8, kh=1, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 0, 0]),
    # as "shallow", "row" and "pointwise_strided", with windows of more than 64 bytes
    "shallow_wide": dict(n=2, c=3, h=11, w=17, oc=33, kh=5, kw=5, stride=[1, 1], dil=[1, 1], pad=[2, 2, 2, 2]),
    "pointwise_strided_deep": dict(n=2, c=83, h=15, w=13, oc=32, kh=1, kw=1, stride=[2, 2], dil=[1, 1], pad=[0, 0, 0, 0]),
    "row_deep": dict(n=2, c=44, h=1, w=61, oc=8, kh=1, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 0, 0]),
}
# quantized windows of at most 64 bytes and quantized 1 x 1 layers are taken by kernels that are asked before the tiles
EARLIER = {"shallow": "conv2d_im2col_i8", "row": "conv2d_im2col_i8", "pointwise_strided": "conv2d_im2col_i8", "pointwise": "pwconv_reg_i8"}


@pytest.mark.parametrize("mode", ["u8", "i8pc", "f16", "f32"])
@pytest.mark.parametrize("name", CASES)
def test_conv2d_tile(oracle, name, mode, monkeypatch):
    rng = np.random.default_rng(list(CASES).index(name) + 400)
    x, wt, b, kws = conv_case(rng, mult=0, mode=mode, **CASES[name])
    monkeypatch.setenv("TVX_CONV_TILE", "1")
    monkeypatch.setenv("TVX_PWCONV_F16", "0")   # (asked before the tiles)
    want = oracle.conv2d(x, wt, b, act=1, **kws)
    assert len(np.unique(want)) > 4
    kernel = EARLIER.get(name, KERNEL[mode]) if mode in ("u8", "i8pc") else KERNEL[mode]
    ran = 0
    for shape in SHAPES:
        monkeypatch.setenv("TVX_CONV_TILE_SHAPE", str(shape))
        got = TC.gpu_conv2d(x, wt, b, act=1, want_kernel=kernel, **kws)
        if mode in ("u8", "i8pc"):
            assert np.array_equal(got, want), (shape, int((got != want).sum()))
        else:
            tol = 2e-3 if mode == "f16" else 1e-5
            scale = np.sqrt(np.mean(want.astype(np.float64) ** 2))
            assert np.abs(got.astype(np.float64) - want).max() <= tol * max(scale, 1.0) * 4, shape
        ran += 1
    assert ran == len(SHAPES)


def test_conv2d_tile_keeps_an_infinity_apart(oracle, monkeypatch):
    """Padding channels and the empty half of an odd last step multiply zero weights: never with another element's infinity."""
    monkeypatch.setenv("TVX_CONV_TILE", "1")
    rng = np.random.default_rng(7)
    for mode in ("f16", "f32"):
        x, wt, b, kws = conv_case(rng, mult=0, mode=mode, n=1, c=3, h=9, w=9, oc=8, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1])
        x[40] = np.inf
        got = TC.gpu_conv2d(x, np.abs(wt) + wt.dtype.type(0.01), b, want_kernel=KERNEL[mode], **kws)
        assert not np.isnan(got).any() and np.isinf(got).sum() == 8 * 9


@pytest.mark.parametrize("mode", ["u8", "i8pc", "f16", "f32"])
@pytest.mark.parametrize("cols", [0, 7, 9])
@pytest.mark.parametrize("groups", [1, 2])
def test_conv2d_tile_blocks_over_one_window(oracle, groups, cols, mode, monkeypatch):
    """Several blocks of output channels over one staged window: an even split, a short last pass, a last block of few channels;
    runs of a whole tile (cols 0: whatever the cost decides, else rows of 7 or 9: no whole quads)."""
    rng = np.random.default_rng(500 + groups + cols)
    x, wt, b, kws = conv_case(rng, mult=0, mode=mode, n=2, c=20 * groups, h=13, w=17, oc=230 if groups == 1 else 140, kh=3, kw=3, stride=[1, 1],
                              dil=[1, 1], pad=[1, 1, 1, 1], **(dict(groups=groups) if groups > 1 else {}))
    monkeypatch.setenv("TVX_CONV_TILE", "1")
    if cols:
        monkeypatch.setenv("TVX_CONV_TILE_COLS", str(cols))
    want = oracle.conv2d(x, wt, b, act=1, **kws)
    for shape, channels in ((0, 64), (2, 64), (4, 32)):
        for loop in (1, 2, 3, 4):
            if loop > -(-kws["out_shape"][2] // groups // channels) or (loop > 1 and shape == 0 and mode == "f32"):
                continue   # (256 x 64 float32 results do not fit LDS beside a window)
            monkeypatch.setenv("TVX_CONV_TILE_SHAPE", str(shape))
            monkeypatch.setenv("TVX_CONV_TILE_LOOP", str(loop))
            got = TC.gpu_conv2d(x, wt, b, act=1, want_kernel=KERNEL[mode], **kws)
            if mode in ("u8", "i8pc"):
                assert np.array_equal(got, want), (shape, loop, int((got != want).sum()))
            else:   # 32-bit sums in another order, rounded to the type (as above)
                scale = max(np.sqrt(np.mean(want.astype(np.float64) ** 2)), 1.0)
                assert np.abs(got.astype(np.float64) - want).max() <= (2e-3 if mode == "f16" else 1e-5) * scale * 4, (shape, loop)


@pytest.mark.parametrize("groups", [1, 3])
@pytest.mark.parametrize("act", [0, 1])
def test_conv2d_tile_rounds_ties_to_even(oracle, act, groups, monkeypatch):
    """Multipliers of .25 to 2 (powers of two among them) on small codes: accumulators shifted up, ties everywhere, exact."""
    rng = np.random.default_rng(600 + groups)
    n, c, h, w, oc = 2, 21, 11, 13, 66
    x, wt = rng.integers(-4, 4, n * c * h * w).astype(np.int8), rng.integers(-4, 4, oc * (c // groups) * 9).astype(np.int8)
    b = rng.integers(-30, 31, oc).astype(np.int32)
    scales = np.array([0.25, 0.5, 0.31, 1.0, 1.7, 0.75])[np.arange(oc) % 6].astype(np.float32)
    kws = dict(in_shape=[w, h, c, n], w_shape=[3, 3, c // groups, oc], out_shape=[w, h, oc, n], stride=[1, 1], dilation=[1, 1], pad_left=1, pad_top=1,
               multiplier=0, in_dtype=1, w_dtype=1, out_dtype=1, in_q=(1.0, -2), w_q=(1.0, 0, scales), out_q=(1.0, 3), **(dict(groups=groups) if groups > 1 else {}))
    monkeypatch.setenv("TVX_CONV_TILE", "1")
    want = oracle.conv2d(x, wt, b, act=act, **kws)
    assert len(np.unique(want)) > 20
    for shape in SHAPES:
        monkeypatch.setenv("TVX_CONV_TILE_SHAPE", str(shape))
        got = TC.gpu_conv2d(x, wt, b, act=act, want_kernel="conv2d_tile_i8", **kws)
        assert np.array_equal(got, want), (shape, int((got != want).sum()))


def _check(got, want, mode, what):
    if mode in ("u8", "i8pc"):
        assert np.array_equal(got, want), (what, int((got != want).sum()))
    else:   # 32-bit sums in another order, rounded to the type (as above)
        scale = max(np.sqrt(np.mean(want.astype(np.float64) ** 2)), 1.0)
        assert np.abs(got.astype(np.float64) - want).max() <= (2e-3 if mode == "f16" else 1e-5) * scale * 4, what


@pytest.mark.parametrize("mode", ["u8", "i8pc", "f16", "f32"])
@pytest.mark.parametrize("k,stride,dil,h,w", [(2, 2, 1, 7, 4), (3, 1, 1, 6, 6), (3, 1, 2, 5, 9), (1, 1, 1, 4, 13), (5, 3, 1, 7, 7)])
def test_conv2d_tile_pads_wider_than_the_window(oracle, k, stride, dil, h, w, mode, monkeypatch):
    """Padding one to four columns (rows) wider than the window: tiles whose window lies left of (above) the image hold nothing but
    padding, whichever way the output columns are cut into tiles."""
    monkeypatch.setenv("TVX_CONV_TILE", "1")
    reach = (k - 1) * dil + 1
    for more in (1, 2, 3, 4):
        rng = np.random.default_rng(700 + 10 * k + more)
        x, wt, b, kws = conv_case(rng, mult=0, mode=mode, n=3, c=20 if k > 1 else 70, h=h, w=w, oc=40, kh=k, kw=k, stride=[stride, stride], dil=[dil, dil],
                                  pad=[reach + more, reach - 1, reach + more if more % 2 else 0, reach - 1])
        want = oracle.conv2d(x, wt, b, act=1, **kws)
        ow = kws["out_shape"][0]
        for cols in sorted({0, ow, (ow + 1) // 2, (ow + 2) // 3} | ({8} if ow >= 8 else set())):
            if cols:
                monkeypatch.setenv("TVX_CONV_TILE_COLS", str(cols))
            else:
                monkeypatch.delenv("TVX_CONV_TILE_COLS", raising=False)
            _check(TC.gpu_conv2d(x, wt, b, act=1, want_kernel=KERNEL[mode], **kws), want, mode, (more, cols))


@pytest.mark.parametrize("mode,case", [("f32", dict(n=4, c=32, h=7, w=4, oc=128, kh=2, kw=2, stride=[2, 2], dil=[1, 1], pad=[3, 0, 0, 0])),
                                       ("i8pc", dict(n=1, c=64, h=6, w=6, oc=128, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[7, 0, 0, 0]))])
def test_conv2d_pads_wider_than_the_window_by_default(oracle, mode, case):
    x, wt, b, kws = conv_case(np.random.default_rng(710), mult=0, mode=mode, **case)
    _check(TC.gpu_conv2d(x, wt, b, act=1, want_kernel=KERNEL[mode], **kws), oracle.conv2d(x, wt, b, act=1, **kws), mode, "default")


ROUTES = [
    # mode, layer, kernel: both sides of the lines between the tiles and the kernels asked behind them, as a caller gets them
    ("u8", dict(c=16, h=8, w=8, oc=16, kh=3, kw=3, pad=[1, 1, 1, 1]), "conv2d_igemm_i8"),            # one granule, weights with a zero point
    ("u8", dict(c=17, h=8, w=8, oc=16, kh=3, kw=3, pad=[1, 1, 1, 1]), "conv2d_tile_i8"),
    ("i8pc", dict(c=16, h=8, w=8, oc=16, kh=3, kw=3, pad=[1, 1, 1, 1]), "conv2d_tile_i8"),           # without one
    ("u8", dict(c=16, h=17, w=17, oc=16, kh=3, kw=3, pad=[1, 1, 1, 1]), "conv2d_tile_i8"),           # rows of no whole dwords, a larger plane
    ("u8", dict(c=16, h=17, w=20, oc=16, kh=3, kw=3, pad=[1, 1, 1, 1]), "conv2d_igemm_i8"),
    ("i8pc", dict(c=80, h=9, w=9, oc=64, kh=1, kw=1, pad=[0] * 4, groups=2), "conv2d_gemm_i8"),      # 32 results of a group
    ("i8pc", dict(c=80, h=9, w=9, oc=66, kh=1, kw=1, pad=[0] * 4, groups=2), "conv2d_tile_i8"),
    ("i8pc", dict(c=8, h=9, w=9, oc=64, kh=1, kw=1, pad=[0] * 4, groups=2), "conv2d_generic"),       # four products a result
    ("i8pc", dict(c=18, h=9, w=9, oc=64, kh=1, kw=1, pad=[0] * 4, groups=2), "conv2d_tile_i8"),
    ("f16", dict(c=64, h=10, w=10, oc=512, kh=1, kw=1, pad=[0] * 4), "pwconv_reg_f16"),              # (1x1 at unit stride: asked before both)
    ("f16", dict(c=64, h=10, w=10, oc=513, kh=1, kw=1, pad=[0] * 4), "pwconv_reg_f16"),
    ("f16", dict(c=32, h=9, w=9, oc=8, kh=1, kw=1, pad=[0] * 4), "pwconv_reg_f16"),
    ("f16", dict(c=144, h=64, w=128, oc=24, kh=1, kw=1, pad=[0] * 4), "pwconv_reg_f16"),
    ("f16", dict(c=144, h=63, w=127, oc=24, kh=1, kw=1, pad=[0] * 4), "pwconv_reg_f16"),
]


@pytest.mark.parametrize("mode,layer,kernel", ROUTES)
def test_conv2d_tile_or_an_older_kernel(oracle, mode, layer, kernel):
    x, wt, b, kws = conv_case(np.random.default_rng(720), mult=0, mode=mode, n=2, stride=[1, 1], dil=[1, 1], **layer)
    got = TC.gpu_conv2d(x, wt, b, act=1, want_kernel=kernel, **kws)
    _check(got, oracle.conv2d(x, wt, b, act=1, **kws), mode, kernel)
