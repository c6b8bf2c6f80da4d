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
