"""The fused MobileNet kernels with four and with eight wavefronts a workgroup, whichever their own rule would take: every block
and pair of the two kernels' test lists, uint8 with the residual Add as second operand, against the oracle (exact)."""
import pytest

import test_gpu_dwpw as DP
import test_gpu_mbconv as MB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("ci", range(len(DP.CASES)))
def test_depthwise_pointwise(oracle, monkeypatch, ci, waves):
    monkeypatch.setenv("TVX_DWPW_WAVES", str(waves))
    DP.test_depthwise_pointwise_fused(oracle, ci, "u8", 2)


@pytest.mark.parametrize("waves", [4, 5, 8])
@pytest.mark.parametrize("ci", range(len(MB.CASES)))
def test_inverted_residual(oracle, monkeypatch, ci, waves):
    monkeypatch.setenv("TVX_MBCONV_WAVES", str(waves))
    MB.test_inverted_residual_block(oracle, ci, "u8", 2, monkeypatch)
