"""A Gaussian-beam step that stops on a negative ce: every workgroup of the
solute kernel that has started finishes its cells, the cells that wait for the
exact temperature included, so a field holds what the whole step gives or what
its buffer held before, bit for bit, and never anything else.  One block, a
batch whose other domain goes on, and coupled ranks, which all stop."""
import numpy as np
import pytest

from mumatscale_amd import abi

pytestmark = pytest.mark.gpu

DIMS = (70, 37, 21)
FIELDS = (abi.FIELD_CL, abi.FIELD_FS, abi.FIELD_GR)
BAD = (10, 18, 33)                                   # z, y, x of the cell with a negative ce
T0 = 20                                              # before the beam turns on: half-solid cells grow, none melts


def _cfg(dims=DIMS):
    from mumatscale_amd.workloads import am_track_config
    cfg = am_track_config(*dims)
    cfg.cell_size, cfg.dt = 1.0e-6, 2.0e-6
    cfg.laser.update(power=60.0, speed=0.8, spot=130e-6, hatch=9e-6, sub_init_temp=600.0,
                     start=[0.0, dims[1] * 0.5e-6, dims[2] * 1.0e-6])
    return cfg


def _substrate(cfg, seed=5):
    """Grain records, gr and fs of a solid block with every third cell half solid."""
    from mumatscale_amd.workloads import voronoi_substrate
    gr, recs = voronoi_substrate(cfg, 40, seed)
    fs = np.zeros(gr.shape)
    fs[1:-1, 1:-1, 1:-1] = np.where(np.random.default_rng(seed).random(gr[1:-1, 1:-1, 1:-1].shape) < 0.3, 0.5, 1.0)
    return recs, gr, fs


def _bad_ce(shape, c_init):
    ce = np.full(shape, c_init)
    ce[BAD] = -1.0
    return ce


def _inner(a):
    return a[1:-1, 1:-1, 1:-1]


def _check(before, whole, got, tile_rows):
    """Every cell from the step or as before it; the tile of the bad cell from the step."""
    done = np.zeros(_inner(before[1]).shape, bool)
    for b, w, g in zip(before, whole, got):
        b, w, g = _inner(b), _inner(w), _inner(g)
        assert np.all((g == w) | (g == b))
        done |= (g == w) & (w != b)
        if tile_rows:
            j0 = (BAD[1] - 1) // tile_rows * tile_rows
            rows = (slice(None), slice(j0, j0 + tile_rows), slice(0, 64))
            assert np.array_equal(g[rows], w[rows])
    assert done.any()


@pytest.mark.parametrize("shape", [(21, 4), (21, 8), (0, 4)], ids=["rows4", "rows8", "cells"])
@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32DEV], ids=["fp64", "fp32"])
def test_block_stopped_by_negative_ce(prec, shape):
    from mumatscale_amd.lib import Subblock
    cfg = _cfg()
    recs, gr, fs = _substrate(cfg)
    got = []
    for check in (False, True):
        with Subblock(cfg.params(check_negative_ce=check, precision=prec), cfg.nucleation()) as sb:
            sb.set_tuning(abi.TUNE_ZM_PLANES, shape[0])
            sb.set_tuning(abi.TUNE_ZM_ROWS, shape[1])
            sb.set_grains(recs)
            sb.upload(abi.FIELD_GR, gr)
            sb.upload(abi.FIELD_FS, fs)
            sb.timestep = T0
            sb.upload(abi.FIELD_CE, _bad_ce(gr.shape, cfg.c_init))
            if not check:
                before = [sb.download(f) for f in FIELDS]
            rep = sb.step(6 if check else 1, raise_on_error=False)
            got.append([sb.download(f) for f in FIELDS])
            if check:
                assert rep.status == abi.ERR_NEGATIVE_CE and rep.failed_step == T0 + 1
                assert abs(sb.solid_volume() / cfg.cell_size ** 3 / _inner(got[1][1]).sum() - 1) < 1e-12
    _check(before, got[0], got[1], shape[1] if shape[0] else 0)


@pytest.mark.parametrize("graph", [0, 1], ids=["launches", "graph"])
@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32DEV], ids=["fp64", "fp32"])
def test_domain_of_a_batch_stopped_by_negative_ce(prec, graph):
    from mumatscale_amd.lib import Batch
    cfgs = [_cfg(), _cfg((65, 18, 30))]
    out = []
    for check in (False, True):
        with Batch([c.params(check_negative_ce=check, precision=prec) for c in cfgs],
                   [c.nucleation() for c in cfgs]) as bt:
            bt.set_tuning(abi.TUNE_ZM_PLANES, 21)
            bt.set_tuning(abi.TUNE_ZM_ROWS, 4)
            bt.set_tuning(abi.TUNE_GRAPH, graph)
            for d, (sb, c) in enumerate(zip(bt.domains, cfgs)):
                recs, gr, fs = _substrate(c, 5 + d)
                sb.set_grains(recs)
                sb.upload(abi.FIELD_GR, gr)
                sb.upload(abi.FIELD_FS, fs)
                sb.timestep = T0
            sb = bt.domains[0]
            sb.upload(abi.FIELD_CE, _bad_ce(sb.shape, cfgs[0].c_init))
            if not check:
                before = [sb.download(f) for f in FIELDS]
                bt.step(1)
                out.append([sb.download(f) for f in FIELDS])
                bt.step(6)                           # to the other domain's last step
            else:
                reps = bt.step(7, raise_on_error=False)
                assert [r.status for r in reps] == [abi.ERR_NEGATIVE_CE, abi.OK]
                out.append([sb.download(f) for f in FIELDS])
            out.append([bt.domains[1].download(f) for f in FIELDS])
    _check(before, out[0], out[2], 4)
    for a, b in zip(out[1], out[3]):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


def test_coupled_ranks_stopped_by_negative_ce():
    from mumatscale_amd.lib import Batch
    cfg = _cfg((70, 74, 21))
    cfg.nsub, cfg.sbdim = [1, 2, 1], [70, 37, 21]
    _, gr, fs = _substrate(_cfg())
    out, before = [], []
    for check in (False, True):
        params = [cfg.params(whole_domain=False, sb_coords=(0, r, 0), check_negative_ce=check) for r in range(2)]
        with Batch(params, [cfg.nucleation(rank=r) for r in range(2)]) as bt:
            for sb in bt.domains:
                sb.upload(abi.FIELD_GR, gr)          # no liquid, so no grain is read
                sb.upload(abi.FIELD_FS, fs)
                sb.timestep = T0
            bt.domains[0].upload(abi.FIELD_CE, _bad_ce(gr.shape, cfg.c_init))
            bt.couple(cfg.nsub)
            if not check:
                before = [[sb.download(f) for f in FIELDS] for sb in bt.domains]
            reps = bt.step(6 if check else 1, raise_on_error=False)
            assert all(r.status == (abi.ERR_NEGATIVE_CE if check else abi.OK) for r in reps)
            out.append([[sb.download(f) for f in FIELDS] for sb in bt.domains])
    for d in range(2):
        _check(before[d], out[0][d], out[1][d], 0)


@pytest.mark.parametrize("why", [abi.ERR_NEGATIVE_CE, abi.ERR_COURANT], ids=["negative_ce", "courant"])
def test_temperature_of_a_stopped_block(why):
    """The separable temperature output, within 1e-13 of the quadrature, at
    the timestep a block has stopped at."""
    from mumatscale_amd.lib import Subblock
    cfg = _cfg()
    recs, gr, fs = _substrate(cfg)
    params = cfg.params(check_negative_ce=True, precision=abi.PREC_FP32DEV)
    if why == abi.ERR_COURANT:
        params.courant_limit = 1.0e-9
    with Subblock(params, cfg.nucleation()) as sb:
        sb.set_grains(recs)
        sb.upload(abi.FIELD_GR, gr)
        sb.upload(abi.FIELD_FS, fs)
        sb.timestep = 70                             # the beam is on, inside the block
        sb.upload(abi.FIELD_CE, _bad_ce(gr.shape, cfg.c_init))
        assert sb.step(3, raise_on_error=False).status == why
        assert sb.get_tuning(abi.TUNE_BEAM_SEP) == 1
        got = sb.download(abi.FIELD_TEMP)
        sb.set_tuning(abi.TUNE_BEAM_SEP, 0)
        want = sb.download(abi.FIELD_TEMP)
    assert want.max() > 1000.0
    assert np.all(np.abs(got - want) <= 1.0e-13 * np.abs(want))
