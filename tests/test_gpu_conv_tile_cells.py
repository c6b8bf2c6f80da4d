"""The tile kernel's staging order, four cells of a plane and then the granules beside them: windows of one to nine cells (none of them
whole fours but two), one to seven granules of channels with and without a partial last one. Against the oracle."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_conv_tile import KERNEL, _check
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["u8", "i8pc", "f16", "f32"])
@pytest.mark.parametrize("h,w", [(1, 8), (2, 7), (3, 5), (4, 8), (5, 6), (3, 16), (7, 8), (9, 4)])
def test_cells(oracle, monkeypatch, h, w, mode):
    monkeypatch.setenv("TVX_CONV_TILE", "1")
    granule = {"u8": 16, "i8pc": 16, "f16": 8, "f32": 4}[mode]
    for c in (granule + 1, 2 * granule, 5 * granule - 3, 7 * granule):
        rng = np.random.default_rng(9000 + 100 * h + 10 * w + c)
        x, wt, b, kws = conv_case(rng, n=3, c=c, h=h, w=w, oc=33, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1], mult=0, mode=mode)
        want = oracle.conv2d(x, wt, b, act=1, **kws)
        for shape in (0, 4, 7):
            monkeypatch.setenv("TVX_CONV_TILE_SHAPE", str(shape))
            _check(TC.gpu_conv2d(x, wt, b, act=1, want_kernel=KERNEL[mode], **kws), want, mode, (c, shape))
