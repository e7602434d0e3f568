"""The Gaussian beam's step evaluates the quadrature only for the cells whose
branch depends on its exact value, from an approximate temperature with an
error bound.  Against the recorded step, which evaluates it in place for every
solid cell (FP64, bit for bit): beams whose time range needs few, many and all
interpolation points, and blocks in which every cell waits for the exact value
(more than a tile's buffer holds)."""
import numpy as np
import pytest

from mumatscale_amd import abi

pytestmark = pytest.mark.gpu

FIELDS = (abi.FIELD_CE, abi.FIELD_CL, abi.FIELD_FS, abi.FIELD_GR, abi.FIELD_DC)
#         name: speed, spot, power, diffusivity factor, fs of the substrate
BEAMS = {"fast": (0.8, 130e-6, 60.0, 1.0, 1.0), "narrow": (0.5, 30e-6, 12.0, 1.0, 1.0),
         "slow_all_nodes": (0.05, 20e-6, 4.0, 1.0, 1.0), "mushy": (0.8, 130e-6, 20.0, 1.0, 0.5)}


@pytest.mark.parametrize("tracks", [1, 2])
@pytest.mark.parametrize("name", list(BEAMS))
def test_beam_step_matches_quadrature_in_place(name, tracks):
    import torch
    from mumatscale_amd.adjoint import record_bytes
    from mumatscale_amd.lib import Subblock
    from mumatscale_amd.workloads import am_track_config, voronoi_substrate
    speed, spot, power, _, fs0 = BEAMS[name]
    cfg = am_track_config(70, 37, 21)
    cfg.cell_size, cfg.dt = 1.0e-6, 2.0e-6
    cfg.am_tracks = tracks
    cfg.laser.update(power=power, speed=speed, spot=spot, hatch=9e-6, sub_init_temp=600.0,
                     start=[0.0, 37e-6 / 2, 21e-6])
    gr, recs = voronoi_substrate(cfg, 40, 5)
    fs = np.zeros(gr.shape)
    fs[1:-1, 1:-1, 1:-1] = fs0
    steps = 140
    out = []
    for recorded, shape in ((True, None), (False, None), (False, (16, 8)), (False, (0, 4))):
        with Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as sb:
            sb.set_grains(recs)
            sb.upload(abi.FIELD_GR, gr)
            sb.upload(abi.FIELD_FS, fs)
            if shape:
                sb.set_tuning(abi.TUNE_ZM_PLANES, shape[0])
                sb.set_tuning(abi.TUNE_ZM_ROWS, shape[1])
            if recorded:
                codes = torch.zeros((steps, record_bytes(sb.params)), dtype=torch.uint8, device="cuda")
                torch.cuda.synchronize()
                sb.set_record(codes.data_ptr(), steps)
            sb.step(steps)
            out.append([sb.download(f) for f in FIELDS])
    want = out[0]
    assert (want[3][1:-1, 1:-1, 1:-1] <= 0).any() or fs0 < 1        # the beam melted something
    assert not np.array_equal(want[2], fs)
    for got in out[1:]:
        for f, a, b in zip(FIELDS, got, want):
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (name, f)
