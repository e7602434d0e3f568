"""Tile edges of the z-marching solute kernel: blocks whose sides are one less
than, equal to and one more than a wave's width, a wave's rows and a walk's
planes, and blocks of a single row or plane, against the cell-parallel kernel
bit for bit (FP64 and FP32-deviation storage, walled and wrapped faces)."""
import numpy as np
import pytest

from mumatscale_amd import abi

pytestmark = pytest.mark.gpu

FIELDS = (abi.FIELD_CE, abi.FIELD_CL, abi.FIELD_FS, abi.FIELD_GR, abi.FIELD_DC)
DIMS = [(63, 7, 15), (64, 8, 16), (65, 9, 17), (1, 1, 40), (129, 1, 2), (2, 33, 1)]


@pytest.mark.parametrize("wall", [1, 0], ids=["walls", "wrapped"])
@pytest.mark.parametrize("prec", [abi.PREC_FP64, abi.PREC_FP32DEV], ids=["fp64", "fp32"])
@pytest.mark.parametrize("dims", DIMS, ids=["x".join(map(str, d)) for d in DIMS])
def test_tiles_match_the_cell_parallel_kernel(dims, prec, wall):
    import bench
    from mumatscale_amd.lib import Subblock
    cfg = bench.directional_config(*dims)
    cfg.dt *= 0.5
    cfg.bulk_density = 1.0e15           # enough grains in a small block
    # and one seed in the middle, for blocks too small to hold a random site
    cfg.fixed.append(tuple((d // 2 + 0.5) * cfg.cell_size for d in dims) + (20.0, 35.0, 50.0, 0.0))
    cfg.pad_bndy = [wall] * 3
    params = lambda: cfg.params(check_negative_ce=False, precision=prec)  # noqa: E731
    with Subblock(params(), cfg.nucleation()) as ref:
        ref.set_tuning(abi.TUNE_ZM_PLANES, 0)
        ref.step(120)
        want = [ref.download(f) for f in FIELDS]
        assert ref.num_grains > 1
    for planes, rows in ((1, 4), (4, 4), (16, 8), (17, 16), (0, 0)):
        with Subblock(params(), cfg.nucleation()) as sb:
            if planes:                  # the last shape is the default one
                sb.set_tuning(abi.TUNE_ZM_PLANES, planes)
                sb.set_tuning(abi.TUNE_ZM_ROWS, rows)
            sb.step(120)
            for f, w in zip(FIELDS, want):
                got = sb.download(f)
                assert np.array_equal(got.view(np.uint8), w.view(np.uint8)), (planes, rows, f)
