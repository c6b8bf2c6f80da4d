"""Average pooling over whole float planes: planes below, at and above a wavefront and its four sums a lane, the last workgroup partly
empty. Against the mean in float64: the type's rounding of the result, and float32 sums of at most 40 additions in a row."""
import numpy as np
import pytest

import tvx_case as TC

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w", [(4, 8), (7, 7), (8, 8), (1, 65), (16, 16), (15, 17), (16, 17), (40, 60)])
@pytest.mark.parametrize("dt,tol", [(2, 2.0 ** -11), (3, 2.0 ** -18)], ids=["f16", "f32"])
@pytest.mark.parametrize("pool_type", [1, 3])
def test_plane_average(pool_type, dt, tol, h, w):
    T = TC.tvx()
    kind = {1: T.POOL_AVG, 3: T.POOL_AVG_ANDROID}[pool_type]
    n, c = 3, 7
    x = (np.random.default_rng(h * 100 + w).standard_normal(n * c * h * w) + 1.0).astype(TC.NP_OF[dt])
    got = TC.gpu_pool2d(x, in_shape=[w, h, c, n], out_shape=[1, 1, c, n], ksize=[w, h], stride=[1, 1], pad_left=0, pad_top=0, pool_type=kind, dtype=dt)
    planes = x.astype(np.float64).reshape(n * c, h * w)
    assert np.all(np.abs(got.astype(np.float64) - planes.mean(1)) <= tol * np.abs(planes).mean(1) * 2)


def test_plane_average_carries_infinities():
    T = TC.tvx()
    x = np.ones((6, 100), np.float32)
    x[1, 70], x[4, 3] = np.inf, np.nan
    got = TC.gpu_pool2d(x.ravel(), in_shape=[10, 10, 6, 1], out_shape=[1, 1, 6, 1], ksize=[10, 10], stride=[1, 1], pad_left=0, pad_top=0,
                        pool_type=T.POOL_AVG, dtype=3)
    assert np.isinf(got[1]) and np.isnan(got[4]) and np.array_equal(got[[0, 2, 3, 5]], np.ones(4, np.float32))
