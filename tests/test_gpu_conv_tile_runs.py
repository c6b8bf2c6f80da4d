"""Results of the tile kernel leaving in runs around sixteen bytes: planes and rows one pixel short of, at and one beyond it, runs
that begin at any byte, for every tile; and rows further apart than 24-bit places reach. Against the oracle."""
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


@pytest.mark.parametrize("step,kernel", [(2 ** 23 - 1, "tile"), (2 ** 23, "other"), (2 ** 24 + 1, "other")])
def test_strides_of_eight_million_rows(oracle, step, kernel):
    """Two rows of results from two rows of the image, `step` apart."""
    c = 10
    x, wt, b, kws = conv_case(np.random.default_rng(8950), n=1, c=c, h=2, w=1, oc=12, kh=1, kw=1, stride=[1, 1], dil=[1, 1], pad=[0, 0, 0, 0], mult=0, mode="f16")
    want = oracle.conv2d(x, wt, b, act=1, **kws).astype(np.float64)
    far = np.full((c, step + 1), 3, dtype=np.float16)
    far[:, [0, step]] = x.reshape(c, 2)
    kws.update(in_shape=[1, step + 1, c, 1], stride=[1, step])
    names = KERNEL["f16"] if kernel == "tile" else ("conv2d_gemm_f16", "conv2d_generic")
    got = TC.gpu_conv2d(far.ravel(), wt, b, act=1, want_kernel=names, **kws)
    # (ten products in float32, then a rounding to float16: half a unit of its last place, 2^-11)
    assert np.abs(got.astype(np.float64) - want).max() <= 2 ** -10 * max(np.abs(want).max(), 1.0)
