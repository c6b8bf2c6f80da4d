"""Window sums of the tile kernel under a weight zero point, on both sides of the line between its two ways to make them (80
multiplications a wavefront), odd last steps and blocks of channels over one window among them. Against the oracle, exact."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_conv_tile import SHAPES
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c,k", [(3, 5), (128, 3), (129, 3), (145, 3), (48, 7), (290, 5)])
@pytest.mark.parametrize("loop", [0, 2])
def test_window_sums(oracle, monkeypatch, c, k, loop):
    rng = np.random.default_rng(9100 + c + k)
    x, wt, b, kws = conv_case(rng, n=2, c=c, h=9, w=11, oc=130, kh=k, kw=k, stride=[1, 1], dil=[1, 1], pad=[k // 2] * 4, mult=0, mode="u8")
    assert kws["w_q"][1] != 128
    monkeypatch.setenv("TVX_CONV_TILE", "1")
    want = oracle.conv2d(x, wt, b, act=1, **kws)
    for shape in SHAPES if not loop else (0, 2, 4):
        if loop and c == 290:
            continue   # (the window is walked in chunks, one block at a time)
        monkeypatch.setenv("TVX_CONV_TILE_SHAPE", str(shape))
        if loop:
            monkeypatch.setenv("TVX_CONV_TILE_LOOP", str(loop))
        # steps of sixteen bytes of a wavefront, for each of its tiles (two in the first three shapes), shared by those that split them (shape 1)
        steps = (k * k * -(-c // 16) + 1) // 2 * (loop or 1)
        variant = "conv2d_tile_i8_box" if shape < 3 and steps * 2 // (2 if shape == 1 else 1) > 80 else "conv2d_tile_i8_sums"
        got = TC.gpu_conv2d(x, wt, b, act=1, want_kernel="conv2d_tile_i8", want_variant=variant, **kws)
        assert np.array_equal(got, want), (shape, int((got != want).sum()))
