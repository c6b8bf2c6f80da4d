"""Which float16 convolutions stay with conv2d_igemm_f16 (3x3 on many rows of 56 pixels or more), which take their pixels in registers (1x1 at unit
stride), and that the kernels on both sides of the line agree with the oracle."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import FLOAT_RTOL, conv_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layer,kernel", [
    (dict(n=2, c=48, h=10, w=10, oc=16, kh=1, kw=1, pad=[0] * 4), "pwconv_reg_f16"),
    (dict(n=2, c=48, h=10, w=10, oc=17, kh=1, kw=1, pad=[0] * 4), "pwconv_reg_f16"),
    (dict(n=2, c=80, h=9, w=10, oc=17, kh=1, kw=1, pad=[0] * 4), "pwconv_reg_f16"),
    (dict(n=2, c=48, h=10, w=10, oc=16, kh=3, kw=3, pad=[1] * 4), "conv2d_tile_f16"),
    (dict(n=2, c=48, h=128, w=128, oc=16, kh=1, kw=1, pad=[0] * 4), "pwconv_reg_f16"),    # 32768 pixels
    (dict(n=21, c=32, h=56, w=56, oc=8, kh=3, kw=3, pad=[1] * 4), "conv2d_igemm_f16"),
    (dict(n=20, c=32, h=56, w=56, oc=8, kh=3, kw=3, pad=[1] * 4), "conv2d_tile_f16"),     # 62720 pixels
])
def test_route(oracle, layer, kernel):
    x, wt, b, kws = conv_case(np.random.default_rng(730), mult=0, mode="f16", stride=[1, 1], dil=[1, 1], **layer)
    want = oracle.conv2d(x, wt, b, act=1, **kws)
    got = TC.gpu_conv2d(x, wt, b, act=1, want_kernel=kernel, **kws)
    assert np.allclose(got.astype(np.float32), want.astype(np.float32), rtol=FLOAT_RTOL, atol=2e-2)
