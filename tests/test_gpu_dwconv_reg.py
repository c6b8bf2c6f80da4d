"""The depthwise register stencil (float16, float32 and int8 windows of 3x3 and 5x5; strides 1 and 2) at the edges of its column and row
groups: planes narrower and lower than a group, ragged ends, padding on every side and on none, the tensor's first and last
elements, planes that share wavefronts and planes that fill them, every row count."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu

NAME = {"u8": "dwconv_planes_i8", "i8pc": "dwconv_planes_i8", "u8pc": "dwconv_planes_i8", "f16": "dwconv_reg_f16", "f32": "dwconv_reg_f32"}
# (n, c, h, w, pad[l,r,t,b] in units of half the window: 1 is SAME)
GRID = [
    (1, 1, 5, 5, 1),     # one plane: its first and last rows are the tensor's
    (3, 5, 7, 6, 1),     # narrower than eight columns
    (2, 3, 3, 3, 1),     # fewer rows and columns than a group, windows that are mostly padding
    (2, 70, 14, 14, 1),  # planes that share wavefronts, more channels than a wavefront holds
    (2, 3, 30, 33, 1),   # ragged column groups
    (1, 4, 40, 64, 0),   # no padding; whole wavefronts a plane
    (1, 2, 67, 75, 1),
]


@pytest.mark.parametrize("mode", ["u8", "i8pc", "u8pc", "f16", "f32"])
@pytest.mark.parametrize("k,stride", [(3, 1), (3, 2), (5, 1), (5, 2)])
@pytest.mark.parametrize("gi", range(len(GRID)))
def test_depthwise_register_stencil(oracle, gi, k, stride, mode, monkeypatch):
    n, c, h, w, same = GRID[gi]
    pads = [[k // 2] * 4, [0, k // 2, 0, k // 2], [k - 1, 0, 1, k - 1]] if same else [[0, 0, 0, 0]]
    rng = np.random.default_rng(7000 + gi)
    if mode not in ("f16", "f32"):
        monkeypatch.setenv("TVX_DWCONV_REG", "1")  # (of their own accord some quantized 3x3 windows go to another stencil)
        TC.expect_variant(monkeypatch, "dwconv_reg_i8")
    for pad in pads:
        if h + pad[2] + pad[3] < k or w + pad[0] + pad[1] < k:
            continue
        x, wt, b, kws = conv_case(rng, n=n, c=c, h=h, w=w, oc=0, kh=k, kw=k, stride=[stride, stride], dil=[1, 1], pad=pad, mult=1, mode=mode)
        want = oracle.conv2d(x, wt, b, act=2, **kws)
        for rows in ("1", "2", "4"):
            monkeypatch.setenv("TVX_DWCONV_REG_ROWS", rows)
            got = TC.gpu_conv2d(x, wt, b, act=2, want_kernel=NAME[mode], **kws)
            if mode in ("f16", "f32"):
                # at most 25 products of float32 sums, of operands of about 1 and 0.2: a few of float32's 2^-24 on values of about 1; float16
                # results differ where the sum falls on the other side of a rounding boundary: one unit in the last place of values up to 6
                assert np.abs(got.astype(np.float64) - want).max() <= (6 * 2.0 ** -10 if mode == "f16" else 1e-5), (pad, rows)
            else:
                assert np.array_equal(got, want), (pad, rows, int((got != want).sum()))


@pytest.mark.parametrize("mode", ["f16", "f32"])
def test_padding_meets_no_infinite_neighbour(oracle, mode):
    """Elements of the neighbouring rows and planes, read and masked, stay out of the windows at the edges."""
    rng = np.random.default_rng(7100)
    x, wt, b, kws = conv_case(rng, n=2, c=3, h=9, w=11, oc=0, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1], mult=1, mode=mode)
    x[99 * 2:99 * 2 + 11] = np.inf   # the third plane's first row, behind the second plane's last
    x[99 * 4 + 98] = np.nan          # the fifth plane's last element
    got = TC.gpu_conv2d(x, np.abs(wt) + wt.dtype.type(0.01), b, want_kernel=NAME[mode], **kws).reshape(6, 9, 11)
    assert np.isinf(got[2, :2]).all() and np.isfinite(got[2, 2:]).all()
    assert np.isnan(got[4]).sum() == 4 and np.isfinite(got[[0, 1, 3, 5]]).all()


def test_infinite_weights_stay_with_the_kernel_that_skips_padding(oracle):
    rng = np.random.default_rng(7200)
    x, wt, b, kws = conv_case(rng, n=1, c=2, h=6, w=6, oc=0, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1], mult=1, mode="f32")
    wt[0] = np.inf
    got = TC.gpu_conv2d(np.abs(x), wt, b, want_kernel="conv2d_generic", **kws).reshape(2, 6, 6)
    assert np.isfinite(got[0, 0]).all() and np.isinf(got[0, 1:, 1:]).all()


@pytest.mark.parametrize("offset", [1, 6, 8])
@pytest.mark.parametrize("mode", ["u8", "i8pc"])
@pytest.mark.parametrize("c,h,w,k,stride", [(3, 160, 160, 5, 1), (5, 14, 14, 3, 1), (4, 7, 9, 3, 2), (2, 20, 21, 5, 2)])
def test_tensors_at_any_address(oracle, c, h, w, k, stride, mode, offset):
    rng = np.random.default_rng(7300)
    x, wt, b, kws = conv_case(rng, n=2, c=c, h=h, w=w, oc=0, kh=k, kw=k, stride=[stride, stride], dil=[1, 1], pad=[k // 2] * 4, mult=1, mode=mode)
    want = oracle.conv2d(x, wt, b, act=2, **kws)
    got = TC.gpu_conv2d(x, wt, b, act=2, want_kernel="dwconv_planes_i8", want_variant="dwconv_reg_i8", misalign=offset, **kws)
    assert np.array_equal(got, want), int((got != want).sum())


@pytest.mark.parametrize("zw", [0, 1, 64, 127, 129, 255])
@pytest.mark.parametrize("k,stride", [(3, 1), (3, 2), (5, 1), (5, 2)])
def test_weight_zero_points_over_their_range(oracle, k, stride, zw, monkeypatch):
    """Every sign and size of the zero point, 0 too (128 in the signed domain, whose negative no byte holds), on codes at both ends."""
    rng = np.random.default_rng(7400 + zw)
    x, wt, b, kws = conv_case(rng, n=2, c=3, h=22, w=33, oc=0, kh=k, kw=k, stride=[stride, stride], dil=[1, 1], pad=[k // 2] * 4, mult=1, mode="u8")
    x, wt = rng.choice([0, 255], x.shape).astype(np.uint8), rng.choice([0, 1, 254, 255], wt.shape).astype(np.uint8)
    kws.update(w_q=(0.01, zw, None), out_q=(0.15 * k, 3))  # (two standard deviations of the sums fill the codes)
    monkeypatch.setenv("TVX_DWCONV_REG", "1")
    want = oracle.conv2d(x, wt, b, act=0, **kws)
    for rows in ("1", "4"):
        monkeypatch.setenv("TVX_DWCONV_REG_ROWS", rows)
        got = TC.gpu_conv2d(x, wt, b, act=0, want_kernel=NAME["u8"], want_variant="dwconv_reg_i8", **kws)
        assert np.array_equal(got, want), (rows, int((got != want).sum()))
