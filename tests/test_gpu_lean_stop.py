"""Lean steps (FP64, 3 M cells and more) of a batch in which one domain stops on
a negative ce: ce of its liquid cells is their cl wherever the failed step was
finished, and the one before it elsewhere, whatever tile was set on the domain's
own context since the batch last stepped; and the other domain goes on."""
import numpy as np
import pytest

from mumatscale_amd import abi
from mumatscale_amd.lib import Batch, Subblock

pytestmark = pytest.mark.gpu


def _cfg(dims, dt_scale):
    import bench
    cfg = bench.directional_config(*dims)
    cfg.dt *= dt_scale                               # partitioning is unstable at the explicit limit (1)
    for q in range(6):
        cfg.fixed.append(tuple((0.15 + 0.13 * q + 0.02 * a) * d * cfg.cell_size for a, d in enumerate(dims)) +
                         (20.0 * q, 35.0, 50.0, 0.0))
    return cfg


@pytest.mark.parametrize("own", [None, (1, 4), (64, 16)], ids=["same", "own1x4", "own64x16"])
def test_domain_of_a_batch_stopped_by_negative_ce(own):
    cfgs = [_cfg((150, 147, 146), 1.0), _cfg((64, 50, 41), 0.5)]
    with Batch([c.params(check_negative_ce=True) for c in cfgs], [c.nucleation() for c in cfgs]) as a, \
            Subblock(cfgs[0].params(check_negative_ce=False), cfgs[0].nucleation()) as b, \
            Subblock(cfgs[1].params(), cfgs[1].nucleation()) as other:
        a.step(2)
        if own:
            a.domains[0].set_tuning(abi.TUNE_ZM_PLANES, own[0])
            a.domains[0].set_tuning(abi.TUNE_ZM_ROWS, own[1])
        reps = a.step(400, raise_on_error=False)
        assert [r.status for r in reps] == [abi.ERR_NEGATIVE_CE, abi.OK]
        failed = reps[0].failed_step
        assert failed > 4
        for _ in range(failed - 1):
            b.step(1)
        prev = b.download(abi.FIELD_CE)
        b.step(1)
        whole = b.download(abi.FIELD_CL)
        ce, cl, gr = (a.domains[0].download(f) for f in (abi.FIELD_CE, abi.FIELD_CL, abi.FIELD_GR))
        inner = (slice(1, -1),) * 3
        ce, cl, gr, prev, whole = ce[inner], cl[inner], gr[inner], prev[inner], whole[inner]
        liquid = gr <= 0
        done = liquid & (cl == whole) & (whole != prev)
        assert done.any()
        assert np.array_equal(ce[done], cl[done])
        assert np.all((ce == cl)[liquid] | (ce == prev)[liquid])
        other.step(402)
        for f in (abi.FIELD_CE, abi.FIELD_CL, abi.FIELD_FS, abi.FIELD_GR):
            assert np.array_equal(a.domains[1].download(f), other.download(f))
