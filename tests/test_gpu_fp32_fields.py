"""FP32-deviation fields on their way to and from the host."""
import numpy as np
import pytest

from mumatscale_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (62, 3, 4), (33, 20, 9)])
def test_fp32_fields_to_and_from_the_host(dims):
    """Uploads store the FP32 rounding of the deviation from c0, downloads give
    c0 plus it in double: the same bits as on the host."""
    from mumatscale_amd.lib import Subblock
    from mumatscale_amd.workloads import directional_config
    cfg = directional_config(*dims)
    rng = np.random.default_rng(2)
    with Subblock(cfg.params(check_negative_ce=False, precision=abi.PREC_FP32DEV), cfg.nucleation()) as sb:
        for f in (abi.FIELD_CE, abi.FIELD_CL):
            h = cfg.c_init * (1 + 0.3 * rng.standard_normal(sb.shape) ** 3)
            sb.upload(f, h)
            want = cfg.c_init + (h - cfg.c_init).astype(np.float32).astype(np.float64)
            assert np.array_equal(sb.download(f).view(np.uint64), want.view(np.uint64))
