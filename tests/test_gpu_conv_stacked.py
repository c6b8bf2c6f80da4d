"""Convolutions of few output channels whose tiles stand for several output rows each, their channels behind one another: rows that do not
divide, strides, groups, uneven pads, planes narrower than a run's store, several images a tile, chunks of the channels, windows under a
weight zero point (the taps outside a row's own hold that). Against the oracle, exact."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu

CASES = {
    "rows": dict(n=2, c=40, h=23, w=37, oc=8, kh=5, kw=5, stride=[1, 1], dil=[1, 1], pad=[2, 2, 2, 2]),
    "strided": dict(n=1, c=70, h=22, w=31, oc=10, kh=3, kw=5, stride=[2, 2], dil=[1, 1], pad=[1, 2, 0, 1]),
    "grouped": dict(n=3, c=40, h=13, w=18, oc=18, kh=7, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 3, 3], groups=2),
    "images": dict(n=7, c=33, h=7, w=5, oc=16, kh=3, kw=3, stride=[1, 1], dil=[1, 1], pad=[1, 1, 1, 1]),
    "chunks": dict(n=1, c=600, h=11, w=19, oc=9, kh=5, kw=5, stride=[1, 1], dil=[2, 1], pad=[4, 4, 2, 2]),
    "window": dict(n=2, c=17, h=4, w=3, oc=4, kh=7, kw=7, stride=[1, 1], dil=[1, 1], pad=[3, 3, 3, 3]),
}


@pytest.mark.parametrize("mode", ["u8", "i8pc"])
@pytest.mark.parametrize("name", CASES)
def test_stacked_rows(oracle, monkeypatch, name, mode):
    rng = np.random.default_rng(list(CASES).index(name) + 8800)
    case = CASES[name]
    x, wt, b, kws = conv_case(rng, mult=0, mode=mode, **case)
    monkeypatch.setenv("TVX_CONV_TILE", "1")
    want = oracle.conv2d(x, wt, b, act=1, **kws)
    assert len(np.unique(want)) > 4
    ran = 0
    for stack in (2, 3, 4):
        if stack * case["oc"] > 32 * case.get("groups", 1):
            continue
        monkeypatch.setenv("TVX_CONV_TILE_STACK", str(stack))
        for shape in (3, 4, 6, 7):   # (those of 32 channels)
            monkeypatch.setenv("TVX_CONV_TILE_SHAPE", str(shape))
            got = TC.gpu_conv2d(x, wt, b, act=1, want_kernel="conv2d_tile_i8", want_variant="conv2d_tile_i8_stacked" + ("_sums" if mode == "u8" else ""), **kws)
            assert np.array_equal(got, want), (stack, shape, int((got != want).sum()))
            ran += 1
    assert ran >= 4
