"""The shape that mmca_batch_autotune picks for a batch of a few small domains
is not slower than the one the batch has by default."""
import pytest

from mumatscale_amd import abi
from mumatscale_amd.lib import Batch, autotune_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32DEV], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 3])
def test_tuned_shape_against_the_default(n, prec):
    from mumatscale_amd.workloads import directional_config
    cfg = directional_config(40, 36, 44)
    cfg.dt *= 0.5
    params = [cfg.params(check_negative_ce=False, precision=prec)] * n
    nucs = [cfg.nucleation()] * n
    planes, rows, _ = autotune_batch(params, nucs)
    t = {}
    with Batch(params, nucs) as bt:
        bt.step(20)
        for shape in (None, (planes, rows)):
            if shape:
                bt.set_tuning(abi.TUNE_ZM_PLANES, shape[0])
                bt.set_tuning(abi.TUNE_ZM_ROWS, shape[1])
            bt.set_kernel_timing(True)
            best = 1e9
            for _ in range(5):
                bt.step(40)
                best = min(best, bt.kernel_time_ms()[0])
            t[shape] = best
    assert t[(planes, rows)] <= 1.25 * t[None], t    # walks of 8 planes: 1.35
