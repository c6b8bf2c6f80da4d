"""The stride-1 inverted-residual kernel in its two tilings, whichever its own rule would take: short last tiles (odd heights, one
row, four columns of 7, 14 and 28), channel counts that fill no chunk, more wavefronts than chunks, the first and the last bytes of
the input tensor, a depthwise weight zero point at the end of its range. Exact against the oracle's operators."""
import pytest

import test_gpu_mbconv as MB

pytestmark = pytest.mark.gpu

CASES = [
    # n, cin, cexp, cout, h, w, stride
    (1, 5, 33, 17, 1, 14, 1),
    (1, 3, 30, 33, 3, 7, 1),
    (2, 33, 70, 5, 5, 14, 1),
    (1, 64, 96, 65, 2, 28, 1),
    (3, 129, 97, 130, 6, 7, 1),
    (2, 8, 200, 170, 4, 14, 1),
]


@pytest.mark.parametrize("mode", ["u8", "i8pc", "u8zp0"])
@pytest.mark.parametrize("wide", [0, 1])
@pytest.mark.parametrize("ci", range(len(CASES)))
def test_tilings(oracle, monkeypatch, ci, wide, mode):
    monkeypatch.setenv("TVX_MBCONV_WIDE", str(wide))
    monkeypatch.setattr(MB, "CASES", CASES)
    if mode == "u8zp0":
        block = MB._block

        def shifted(*args):
            x, first, (wd, bd, kd), last = block(*args)
            kd["w_q"] = (kd["w_q"][0], 0, None)
            kd["out_q"] = (kd["out_q"][0] * 2, kd["out_q"][1])  # (every tap counts 120-odd more)
            last[2]["in_q"] = kd["out_q"]
            return x, first, (wd, bd, kd), last
        monkeypatch.setattr(MB, "_block", shifted)
    MB.test_inverted_residual_block(oracle, ci, "u8" if mode == "u8zp0" else mode, ci % 3, monkeypatch)


@pytest.mark.parametrize("n,cin,cexp,cout,w,taken", [
    (13, 32, 64, 96, 28, True), (14, 32, 64, 96, 28, False), (5, 128, 160, 32, 28, True), (6, 128, 160, 32, 28, False), (6, 32, 64, 100, 28, False),
    (64, 64, 96, 160, 14, True), (1, 64, 96, 161, 14, False), (64, 64, 96, 160, 7, True), (1, 64, 96, 161, 7, False)])
def test_blocks_taken_of_its_own_accord(n, cin, cexp, cout, w, taken):
    """Both sides of each line of the rule, at 256 compute units."""
    import numpy as np
    import torch
    import tvx_case as TC
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are drawn in workgroups a compute unit")
    T, keep = TC.tvx(), []
    x, (w1, b1, k1), (wd, bd, kd), (w3, b3, k3) = MB._block(np.random.default_rng(3), 1, cin, cexp, cout, w, w, 1, "u8")
    for k in (k1, kd, k3):
        k["in_shape"][3] = k["out_shape"][3] = n
    descs = [MB._desc(T, k, 0, keep) for k in (k1, kd, k3)]
    try:
        T.mbconv_create(descs[0], w1, b1, descs[1], wd, bd, descs[2], w3, b3).close()
    except T.TvxError as e:
        assert e.status == T.E_UNSUPPORTED and not taken
    else:
        assert taken
