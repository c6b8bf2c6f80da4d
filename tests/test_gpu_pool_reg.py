"""The pooling register stencil (2x2 and 3x3 windows at stride 1 or 2, 7x7 windows side by side; every type) at the edges of its
groups of columns and rows: planes narrower and lower than a group, ragged ends, padding on every side and on none, the
tensor's first and last elements."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import rand_q

pytestmark = pytest.mark.gpu

NAME = {0: "pool2d_rows_i8", 1: "pool2d_rows_i8", 2: "pool2d_reg_f16", 3: "pool2d_reg_f32"}
SHAPES = [(7, 5, 3, 2), (4, 9, 1, 1), (15, 14, 70, 2), (33, 30, 3, 1), (68, 41, 2, 2), (9, 8, 40, 3)]   # {W, H, C, N}


def values(rng, n, dtype):
    return rand_q(rng, n, dtype) if dtype < 2 else rng.standard_normal(n).astype(np.float16 if dtype == 2 else np.float32)


@pytest.mark.parametrize("dtype", [0, 1, 2, 3])
@pytest.mark.parametrize("ptype", [0, 1, 3])
@pytest.mark.parametrize("k,s", [(2, 1), (2, 2), (3, 1), (3, 2), (7, 7)])
@pytest.mark.parametrize("si", range(len(SHAPES)))
def test_pool2d_register_stencil(oracle, si, k, s, ptype, dtype, monkeypatch):
    w, h, c, n = SHAPES[si]
    rng = np.random.default_rng(8000 + si * 100 + k * 10 + s)
    zi = 7 if dtype == 1 else 120
    if dtype < 2:
        TC.expect_variant(monkeypatch, "pool2d_reg_i8")
    scales = (((0.1, zi), (0.1, zi)), ((0.1, zi), (0.1, zi - 9)), ((0.1, zi), (0.07, 3))) if dtype < 2 else (((1.0, 0), (1.0, 0)),)
    for pad in ([0, 0, 0, 0], [0, 1, 0, 1], [1, 1, 1, 1], [k - 1, 0, k - 1, k - 1]):
        ow, oh = (w + pad[0] + pad[1] - k) // s + 1, (h + pad[2] + pad[3] - k) // s + 1
        if w + pad[0] + pad[1] < k or h + pad[2] + pad[3] < k or (ow - 1) * s >= w + pad[0] or (oh - 1) * s >= h + pad[2]:
            continue
        if ptype != 0 and ow == 1 and oh == 1 and (w, h) == (k, k):
            continue
        x = values(rng, w * h * c * n, dtype)
        kws = dict(in_shape=[w, h, c, n], out_shape=[ow, oh, c, n], ksize=[k, k], stride=[s, s], pad_left=pad[0], pad_top=pad[2], pool_type=ptype, dtype=dtype)
        for in_q, out_q in scales:
            want = oracle.pool2d(x, in_q=in_q, out_q=out_q, **kws)
            name = "pool2d_reg_i8" if dtype < 2 and k == 7 else NAME[dtype]
            for rows in ("1", "4")[:2 if s == 1 else 1]:
                monkeypatch.setenv("TVX_POOL_REG_ROWS", rows)
                got = TC.gpu_pool2d(x, in_q=in_q, out_q=out_q, want_kernel=name, **kws)
                if dtype < 2 or ptype == 0:
                    assert np.array_equal(got, want), (pad, in_q, out_q, rows, int((got != want).sum()))
                else:
                    # sums of up to 49 normal values in float32, rounded to the type: a unit in the last place of values up to 4
                    assert np.abs(got.astype(np.float64) - want).max() <= (4 * 2.0 ** -10 if dtype == 2 else 4 * 2.0 ** -21), (pad, rows)


@pytest.mark.parametrize("dtype", [2, 3])
def test_max_pool_of_lowest_values_and_infinities(oracle, dtype):
    """Padding never wins, and what the neighbouring rows hold stays out of a window."""
    lowest = -np.finfo(np.float16 if dtype == 2 else np.float32).max
    x = np.full(2 * 9 * 11, lowest, np.float16 if dtype == 2 else np.float32)
    x[99:110] = np.inf      # the second plane's first row
    x[98] = np.nan          # the first plane's last element: no maximum is a NaN
    x[50] = -np.inf
    kws = dict(in_shape=[11, 9, 2, 1], out_shape=[11, 9, 2, 1], ksize=[3, 3], stride=[1, 1], pad_left=1, pad_top=1, pool_type=0, dtype=dtype)
    got = TC.gpu_pool2d(x, want_kernel=NAME[dtype], **kws).reshape(2, 9, 11)
    assert (got[0] == lowest).all() and np.isinf(got[1, :2]).all() and (got[1, 2:] == lowest).all()


@pytest.mark.parametrize("dtype", [0, 1, 2, 3])
@pytest.mark.parametrize("w,h", [(64, 32), (45, 46), (127, 129), (159, 160), (16, 1061)])
def test_average_of_large_planes(oracle, w, h, dtype, monkeypatch):
    """A workgroup per plane: whole units of sixteen bytes and what is left of them, planes that begin at any element."""
    rng = np.random.default_rng(8100 + w)
    c, n = 3, 2
    x = values(rng, w * h * c * n, dtype)
    if dtype > 1:
        x = x + x.dtype.type(1)
    kws = dict(in_shape=[w, h, c, n], out_shape=[1, 1, c, n], ksize=[w, h], stride=[1, 1], pad_left=0, pad_top=0, pool_type=1, dtype=dtype)
    q = dict(in_q=(0.1, 3), out_q=(0.002, 5)) if dtype < 2 else {}
    TC.expect_variant(monkeypatch, "pool2d_plane_sum")
    want = oracle.pool2d(x, **q, **kws)
    got = TC.gpu_pool2d(x, **q, **kws)
    if dtype < 2:
        assert np.array_equal(got, want)
    else:
        # means of about 1 from float32 sums of w h terms of about 1 in another order
        assert np.abs(got.astype(np.float64) - want).max() <= (2.0 ** -10 if dtype == 2 else w * h * 2.0 ** -24)
