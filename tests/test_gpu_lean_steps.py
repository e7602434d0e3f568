"""Steps of one long call, which leave unwritten what stays as it is (blocks
of 3 M cells and more in FP64 storage), against calls of a few steps, which
write everything: bit for bit, over both tile shapes, odd and even numbers of
steps, uploaded states with ce and cl apart, batches with graphs, coupled
ranks, and calls that stop on an error."""
import numpy as np
import pytest

from mumatscale_amd import abi
from mumatscale_amd.lib import Batch, Subblock

pytestmark = pytest.mark.gpu

FIELDS = (abi.FIELD_CE, abi.FIELD_CL, abi.FIELD_FS, abi.FIELD_GR, abi.FIELD_DC)
DIMS = (150, 147, 146)


def _cfg(dims=DIMS, bulk=3.0e13, wall=1):
    import bench
    cfg = bench.directional_config(*dims)
    cfg.dt *= 0.5
    cfg.bulk_density = bulk
    cfg.pad_bndy = [wall] * 3
    for q in range(6):                               # grains from the first steps on
        cfg.fixed.append(tuple((0.15 + 0.13 * q + 0.02 * a) * d * cfg.cell_size for a, d in enumerate(dims)) +
                         (20.0 * q, 35.0, 50.0, 0.0))
    return cfg


def _same(a, b, where):
    for f in FIELDS:
        x, y = a.download(f), b.download(f)
        assert np.array_equal(x.view(np.uint8), y.view(np.uint8)), (where, f)


@pytest.mark.parametrize("wall", [1, 0], ids=["walls", "wrapped"])
@pytest.mark.parametrize("rows", [4, 8, 16])
def test_long_call_matches_short_ones(rows, wall):
    cfg = _cfg(wall=wall)
    rng = np.random.default_rng(rows)
    with Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as a, \
            Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as b:
        for s in (a, b):
            s.set_tuning(abi.TUNE_ZM_PLANES, 16)
            s.set_tuning(abi.TUNE_ZM_ROWS, rows)
        for n in (40, 9, 8, 31):
            a.step(n)
            for q in range(0, n, 5):
                b.step(min(5, n - q))
            assert a.num_grains == b.num_grains
            _same(a, b, n)
            if n == 9:                               # a state no step has left: ce and cl of the liquid differ
                ce = a.download(abi.FIELD_CE)
                ce = ce * (1.0 + 1.0e-6 * rng.random(ce.shape))
                for s in (a, b):
                    s.upload(abi.FIELD_CE, ce)
        assert a.num_grains > 20


@pytest.mark.parametrize("coupled", [False, True], ids=["batch", "coupled"])
def test_batches(coupled):
    if coupled:
        cfg = _cfg((256, 120, 110))
        cfg.nsub, cfg.sbdim = [2, 1, 1], [128, 120, 110]
        params = [cfg.params(whole_domain=False, sb_coords=(r, 0, 0), check_negative_ce=False) for r in range(2)]
        nucs = [cfg.nucleation(rank=r) for r in range(2)]
    else:
        cfgs = [_cfg((150, 147, 100)), _cfg((64, 50, 41), 1.0e15), _cfg((130, 97, 80))]
        params = [c.params(check_negative_ce=False) for c in cfgs]
        nucs = [c.nucleation() for c in cfgs]
    with Batch(params, nucs) as a, Batch(params, nucs) as b:
        if coupled:
            for s in (a, b):
                s.couple(cfg.nsub)
        else:
            a.set_tuning(abi.TUNE_GRAPH, 1)
        for n in (41, 12, 30):
            a.step(n)
            for q in range(0, n, 6):
                b.step(min(6, n - q))
            for x, y in zip(a.domains, b.domains):
                _same(x, y, n)


def test_stopped_by_the_grain_capacity():
    cfg = _cfg(bulk=3.0e15)
    with Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as s:
        s.step(20)
        while True:                                  # a step that creates two grains or more
            before = s.num_grains
            s.step(1)
            if s.num_grains > before + 1:
                break
            assert s.timestep < 200
        failed = s.timestep
    cfg.max_total_grains = before                    # its second grain finds no slot
    with Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as a, \
            Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as b:
        r = a.step(300, raise_on_error=False)
        for _ in range(60):
            q = b.step(5, raise_on_error=False)
            if q.status != abi.OK:
                break
        assert r.status == q.status == abi.ERR_GRAIN_CAPACITY and r.failed_step == q.failed_step == failed
        _same(a, b, r.failed_step)


def test_stopped_by_negative_ce():
    cfg = _cfg()
    cfg.dt *= 2.0                                    # partitioning is unstable at the explicit limit
    with Subblock(cfg.params(check_negative_ce=True), cfg.nucleation()) as a, \
            Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as b:
        r = a.step(400, raise_on_error=False)
        assert r.status == abi.ERR_NEGATIVE_CE and r.failed_step > 2
        # liquid cells of tiles that finished the failed step: ce is their cl;
        # of the other tiles: ce of the step before
        for _ in range(r.failed_step - 1):
            b.step(1)
        ce, cl, gr = a.download(abi.FIELD_CE), a.download(abi.FIELD_CL), a.download(abi.FIELD_GR)
        liquid = np.zeros(gr.shape, bool)
        liquid[1:-1, 1:-1, 1:-1] = gr[1:-1, 1:-1, 1:-1] <= 0
        assert np.all((ce == cl)[liquid] | (ce == b.download(abi.FIELD_CE))[liquid])
