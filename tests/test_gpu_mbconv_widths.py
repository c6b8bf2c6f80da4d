"""The stride-1 inverted-residual kernel on widths that are none of its two-form ones: last column tiles of one to four columns, planes of one
tile, odd heights and a single row, the first and the last bytes of the input tensor. Exact against the oracle's operators."""
import numpy as np
import pytest

import test_gpu_mbconv as MB
import tvx_case as TC

pytestmark = pytest.mark.gpu

CASES = [
    # n, cin, cexp, cout, h, w, stride
    (1, 1, 97, 17, 2, 3, 1),
    (2, 3, 130, 33, 3, 4, 1),
    (3, 33, 128, 5, 5, 5, 1),
    (2, 24, 144, 24, 6, 6, 1),
    (1, 64, 200, 65, 1, 9, 1),
    (2, 96, 100, 96, 7, 10, 1),
    (1, 129, 160, 130, 4, 13, 1),
    (1, 24, 144, 24, 9, 57, 1),
]


@pytest.mark.parametrize("mode", ["u8", "i8pc"])
@pytest.mark.parametrize("ci", range(len(CASES)))
def test_widths(oracle, monkeypatch, ci, mode):
    monkeypatch.setattr(MB, "CASES", CASES)
    for add in range(3):
        MB.test_inverted_residual_block(oracle, ci, mode, add, monkeypatch)


@pytest.mark.parametrize("n,cin,cexp,cout,h,w,taken", [
    (1, 24, 128, 24, 12, 12, True), (1, 24, 96, 24, 12, 12, False), (1, 24, 128, 24, 12, 2, False), (1, 64, 128, 161, 12, 12, False),
    (40, 24, 128, 24, 16, 16, True), (41, 24, 128, 24, 16, 16, False), (16, 128, 128, 32, 16, 16, True), (17, 128, 128, 32, 16, 16, False),
    # many chunks of more than three steps: a second workgroup of a CU just begun, one small image whose planes are whole dwords and whose rows are not
    (33, 160, 960, 160, 8, 8, False), (32, 160, 960, 160, 8, 8, True), (40, 160, 960, 160, 8, 8, True), (33, 160, 768, 160, 8, 8, True), (15, 160, 960, 160, 12, 12, True),
    (4, 128, 768, 128, 24, 24, False), (5, 128, 768, 128, 24, 24, True), (5, 160, 960, 160, 24, 24, False), (7, 160, 960, 160, 24, 24, True),
    (4, 96, 960, 96, 24, 24, True),
    (1, 160, 960, 160, 10, 10, False), (2, 160, 960, 160, 10, 10, True), (1, 160, 800, 160, 10, 10, True), (1, 160, 960, 160, 7, 6, True), (1, 160, 960, 160, 9, 12, True),
    (1, 160, 960, 160, 12, 9, False), (1, 160, 960, 160, 18, 18, True), (1, 160, 960, 160, 14, 14, True), (1, 160, 960, 160, 7, 7, True)])
def test_blocks_taken_by_workgroups(n, cin, cexp, cout, h, w, taken):
    """Both sides of the rule's lines, at 256 compute units."""
    import torch
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are drawn in workgroups a compute unit")
    T, keep = TC.tvx(), []
    x, (w1, b1, k1), (wd, bd, kd), (w3, b3, k3) = MB._block(np.random.default_rng(3), 1, cin, cexp, cout, h, w, 1, "u8")
    for k in (k1, kd, k3):
        k["in_shape"][3] = k["out_shape"][3] = n
    descs = [MB._desc(T, k, 0, keep) for k in (k1, kd, k3)]
    try:
        T.mbconv_create(descs[0], w1, b1, descs[1], wd, bd, descs[2], w3, b3).close()
    except T.TvxError as e:
        assert e.status == T.E_UNSUPPORTED and not taken
    else:
        assert taken
