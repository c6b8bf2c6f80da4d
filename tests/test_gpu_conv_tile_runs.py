"""Results of the tile kernel leaving in runs around sixteen bytes: planes and rows one pixel short of, at and one beyond it, runs
that begin at any byte, for every tile. Against the oracle."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_conv_tile import KERNEL, SHAPES
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["u8", "f16"])
@pytest.mark.parametrize("h,w", [(1, 8), (2, 7), (3, 3), (1, 15), (4, 4), (1, 17), (5, 9), (13, 23), (2, 130)])
def test_runs(oracle, monkeypatch, h, w, mode):
    rng = np.random.default_rng(8900 + 200 * h + w)
    x, wt, b, kws = conv_case(rng, n=3, c=20, h=h, w=w, oc=35, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1], mult=0, mode=mode)
    monkeypatch.setenv("TVX_CONV_TILE", "1")
    want = oracle.conv2d(x, wt, b, act=1, **kws)
    for shape in SHAPES:
        monkeypatch.setenv("TVX_CONV_TILE_SHAPE", str(shape))
        got = TC.gpu_conv2d(x, wt, b, act=1, want_kernel=KERNEL[mode], **kws)
        if mode == "u8":
            assert np.array_equal(got, want), (shape, int((got != want).sum()))
        else:   # (a unit of float16's last place at the results' scale, as the tile kernel's other tests)
            scale = np.sqrt(np.mean(want.astype(np.float64) ** 2))
            assert np.abs(got.astype(np.float64) - want).max() <= 8e-3 * max(scale, 1.0), shape
