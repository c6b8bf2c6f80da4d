"""Convolutions on both sides of the lines between the tiles and the kernels for few products, short windows and pointwise layers: the kernel that
takes them without a lever (at 256 compute units), and its results against the oracle, over odd sizes, strides and uneven padding."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu

P0, P1 = [0] * 4, [1] * 4
LAYERS = [
    # short windows of bytes: a handful of pixels, between, eighty thousand
    ("i8pc", dict(n=2, c=12, h=15, w=16, oc=33, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_im2col_i8"),      # 128 pixels
    ("u8", dict(n=3, c=12, h=15, w=11, oc=33, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_tile_i8"),          # 144
    ("i8pc", dict(n=1, c=43, h=17, w=17, oc=80, kh=1, kw=1, stride=[2, 1], pad=P0), "conv2d_tile_i8"),
    ("u8", dict(n=4, c=1, h=70, w=71, oc=9, kh=7, kw=7, stride=[2, 2], pad=[3, 2, 3, 3]), "conv2d_tile_i8"),  # 4900, of 49 bytes
    ("i8pc", dict(n=2, c=7, h=45, w=45, oc=5, kh=3, kw=3, stride=[1, 1], pad=P1, dil=[2, 1]), "conv2d_im2col_i8"),  # 43 x 45 pixels and dilated rows
    ("u8", dict(n=5, c=8, h=252, w=256, oc=6, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_im2col_i8"),        # 80640
    ("u8", dict(n=5, c=8, h=248, w=255, oc=6, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_tile_i8"),          # 79360
    ("u8", dict(n=1, c=3, h=300, w=301, oc=20, kh=3, kw=3, pad=[16] * 4, dil=[16, 16]), "conv2d_tile_i8"),    # 90300, taps further apart than conv2d_im2col_i8 reaches
    # a granule of channels under weights with a zero point: two million products
    ("u8", dict(n=3, c=16, h=14, w=16, oc=20, kh=3, kw=3, pad=P1), "conv2d_igemm_i8"),
    ("u8", dict(n=3, c=16, h=14, w=16, oc=21, kh=3, kw=3, pad=P1), "conv2d_tile_i8"),
    ("u8", dict(n=2, c=9, h=40, w=44, oc=17, kh=3, kw=3, pad=P1), "conv2d_tile_i8"),
    # floating point, a handful of products an output
    ("f32", dict(n=2, c=1, h=50, w=60, oc=50, kh=1, kw=1, pad=P0), "conv2d_generic"),                          # 300000 outputs
    ("f32", dict(n=2, c=1, h=50, w=60, oc=51, kh=1, kw=1, pad=P0), "conv2d_tile_f32"),
    ("f16", dict(n=2, c=3, h=50, w=50, oc=41, kh=1, kw=1, pad=P0), "pwconv_reg_f16"),                          # (unit stride)
    ("f16", dict(n=2, c=3, h=99, w=99, oc=41, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_tile_f16"),          # 205000
    ("f32", dict(n=1, c=1, h=30, w=41, oc=25, kh=3, kw=3, pad=P1), "conv2d_generic"),                          # 30750 outputs
    ("f16", dict(n=1, c=1, h=29, w=41, oc=25, kh=3, kw=3, pad=P1), "conv2d_generic"),
    ("f32", dict(n=4, c=1, h=30, w=34, oc=25, kh=3, kw=3, pad=P1), "conv2d_generic"),                          # 102000
    ("f16", dict(n=4, c=1, h=30, w=35, oc=25, kh=3, kw=3, pad=P1), "conv2d_tile_f16"),                         # 105000
    ("f32", dict(n=19, c=1, h=144, w=144, oc=1, kh=3, kw=3, pad=[2] * 4, dil=[2, 2]), "conv2d_generic"),       # few channels: of one, three and six
    ("f16", dict(n=4, c=1, h=256, w=257, oc=3, kh=3, kw=3, pad=P1), "conv2d_generic"),
    ("f16", dict(n=4, c=1, h=267, w=257, oc=3, kh=3, kw=3, pad=P1), "conv2d_tile_f16"),
    ("f32", dict(n=3, c=1, h=118, w=119, oc=6, kh=3, kw=3, pad=P1), "conv2d_generic"),
    ("f32", dict(n=3, c=1, h=118, w=122, oc=6, kh=3, kw=3, pad=P1), "conv2d_tile_f32"),
    ("f32", dict(n=3, c=1, h=60, w=62, oc=18, kh=1, kw=5, pad=[2, 2, 0, 0]), "conv2d_generic"),                # 200880 of five products
    ("f32", dict(n=3, c=4, h=60, w=62, oc=18, kh=1, kw=2, pad=[1, 0, 0, 0]), "conv2d_tile_f32"),               # 200880 of eight
    ("f32", dict(n=1, c=8, h=9, w=11, oc=12, kh=1, kw=1, pad=P0), "conv2d_tile_f32"),
    ("f32", dict(n=2, c=4, h=41, w=42, oc=40, kh=1, kw=1, pad=P0), "conv2d_generic"),                          # 137760 of four products
    ("f32", dict(n=2, c=4, h=41, w=43, oc=40, kh=1, kw=1, pad=P0), "conv2d_tile_f32"),                         # 141040
    ("f16", dict(n=2, c=5, h=39, w=63, oc=79, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_generic"),           # 101120 of five
    ("f16", dict(n=2, c=5, h=39, w=63, oc=81, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_tile_f16"),          # 103680
    ("f32", dict(n=2, c=5, h=9, w=11, oc=12, kh=1, kw=1, pad=P0), "conv2d_tile_f32"),
    # float16, pointwise: at unit stride pixels in registers, whatever their number and that of the results
    ("f16", dict(n=2, c=24, h=13, w=13, oc=24, kh=1, kw=1, pad=P0), "pwconv_reg_f16"),
    ("f16", dict(n=2, c=24, h=13, w=13, oc=25, kh=1, kw=1, pad=P0), "pwconv_reg_f16"),
    ("f16", dict(n=3, c=48, h=14, w=14, oc=40, kh=1, kw=1, pad=P0), "pwconv_reg_f16"),
    ("f16", dict(n=1, c=144, h=128, w=128, oc=65, kh=1, kw=1, pad=P0), "pwconv_reg_f16"),
    ("f16", dict(n=2, c=40, h=15, w=17, oc=33, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_tile_f16"),
    # ... strided: few channels and results, results too few for a matrix tile, few results of more channels
    ("f16", dict(n=7, c=24, h=16, w=16, oc=16, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_gemm_f16"),
    ("f16", dict(n=7, c=24, h=16, w=16, oc=7, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_tile_f16"),
    ("f16", dict(n=2, c=32, h=19, w=17, oc=8, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_gemm_f16"),
    ("f16", dict(n=2, c=32, h=19, w=17, oc=9, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_tile_f16"),
    ("f16", dict(n=1, c=48, h=62, w=62, oc=11, kh=1, kw=1, stride=[2, 2], pad=P0), "conv2d_tile_f16"),
]


@pytest.mark.parametrize("mode,layer,kernel", LAYERS)
def test_conv_choice(oracle, mode, layer, kernel):
    x, wt, b, kws = conv_case(np.random.default_rng(740), mult=0, mode=mode, **{"stride": [1, 1], "dil": [1, 1], **layer})
    want = oracle.conv2d(x, wt, b, act=1, **kws)
    got = TC.gpu_conv2d(x, wt, b, act=1, want_kernel=kernel, **kws)
    if mode in ("u8", "i8pc"):
        assert np.array_equal(got, want), int((got != want).sum())
    else:   # a sum's rounding in float32, and that of the result: 2^-11 for float16
        scale = np.sqrt(np.mean(want.astype(np.float64) ** 2))
        assert np.abs(got.astype(np.float64) - want).max() <= (2e-3 if mode == "f16" else 1e-5) * max(scale, 1.0) * 4
