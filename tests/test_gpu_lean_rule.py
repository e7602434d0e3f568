"""Which blocks' calls are lean, as the benchmark's roofline reads it."""
import pytest

from mumatscale_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,prec,planes,want", [((160, 150, 140), abi.PREC_FP64, None, 8),
                                                   ((120, 150, 140), abi.PREC_FP64, None, 0),
                                                   ((160, 150, 140), abi.PREC_FP32DEV, None, 0),
                                                   ((160, 150, 140), abi.PREC_FP64, 0, 0)])
def test_lean_steps_of_a_block(dims, prec, planes, want):
    from mumatscale_amd.lib import Subblock
    from mumatscale_amd.workloads import directional_config
    cfg = directional_config(*dims)
    with Subblock(cfg.params(check_negative_ce=False, precision=prec), cfg.nucleation()) as sb:
        if planes is not None:
            sb.set_tuning(abi.TUNE_ZM_PLANES, planes)
        assert sb.get_tuning(abi.TUNE_LEAN_STEPS) == want
        with pytest.raises(abi.MmcaError):
            sb.set_tuning(abi.TUNE_LEAN_STEPS, 8)
