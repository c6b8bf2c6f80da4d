"""Which kernel takes a quantized depthwise 3x3 layer of rows that are whole dwords, on both sides of the lines by planes, and the four- and
eight-column forms on either side of theirs (at 256 compute units). Exact against the oracle."""
import numpy as np
import pytest

import tvx_case as TC
from test_gpu_parity import conv_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,h,w,stride,kernel", [
    (24, 128, 8, 8, 1, "dwconv_rows_i8"), (23, 128, 8, 8, 1, "dwconv3x3_i8"),
    (6, 1000, 16, 16, 1, "dwconv_rows_i8"), (6, 999, 16, 16, 1, "dwconv3x3_i8"),
    (12, 1000, 20, 20, 1, "dwconv_rows_i8"), (12, 1000, 21, 20, 1, "dwconv3x3_i8"),
    (4, 1000, 16, 16, 2, "dwconv_rows_i8"), (6, 1000, 32, 32, 2, "dwconv_rows_i8"), (6, 999, 32, 32, 2, "dwconv3x3_i8"),
    (2, 3, 9, 56, 1, "dwconv3x3_i8"), (1, 5, 9, 88, 1, "dwconv3x3_i8"), (1, 5, 9, 96, 1, "dwconv3x3_i8"),
    # tall planes
    (2, 3, 95, 16, 1, "dwconv3x3_i8"), (1, 3, 96, 16, 1, "dwconv3x3_i8_eight"), (1, 2, 130, 224, 1, "dwconv3x3_i8_eight"), (2, 3, 97, 20, 1, "dwconv3x3_i8"),
    (2, 3, 192, 16, 2, "dwconv3x3_i8"),
    # wavefronts of a plane with four and eight columns, without window sums (even batches) and with them: two and one, four and two, three and two, ten and five
    (2, 255, 24, 40, 1, "dwconv3x3_i8"), (2, 256, 24, 40, 1, "dwconv3x3_i8_eight"), (23, 133, 24, 40, 1, "dwconv3x3_i8"), (23, 134, 24, 40, 1, "dwconv3x3_i8_eight"),
    (16, 143, 53, 56, 1, "dwconv3x3_i8"), (16, 144, 53, 56, 1, "dwconv3x3_i8_eight"), (15, 153, 53, 56, 1, "dwconv3x3_i8"), (15, 154, 53, 56, 1, "dwconv3x3_i8_eight"),
    (40, 192, 45, 48, 1, "dwconv3x3_i8"), (8, 115, 78, 80, 1, "dwconv3x3_i8"), (8, 116, 78, 80, 1, "dwconv3x3_i8_eight"), (5, 511, 78, 80, 1, "dwconv3x3_i8"),
    (5, 512, 78, 80, 1, "dwconv3x3_i8_eight")])
def test_depthwise_choice(oracle, n, c, h, w, stride, kernel):
    pad = [1, 1, 1, 1] if stride == 1 else [0, 1, 0, 1]
    rng = np.random.default_rng(9500 + h * w + n)
    x, wt, b, kws = conv_case(rng, n=n, c=c, h=h, w=w, oc=0, kh=3, kw=3, stride=[stride, stride], dil=[1, 1], pad=pad, mult=1, mode="u8" if n % 2 else "i8pc")
    got = TC.gpu_conv2d(x, wt, b, act=2, want_variant=kernel, **kws)
    assert np.array_equal(got, oracle.conv2d(x, wt, b, act=2, **kws))
