"""Interface list and nucleation at the sizes where their launches change:
mask words at a list workgroup's edges (64 and 256 words), either side of the
largest list whose counts are scanned in the counting launch (192 workgroups of
256 words) and of the largest one written 64 words at a time (2048 workgroups),
against the list of the gr field by numpy; and one, two and three detecting
workgroups of 256 nucleation sites against the single operators."""
import numpy as np
import pytest

from mumatscale_amd import abi

pytestmark = pytest.mark.gpu


def _cfg(*dims):
    import bench
    cfg = bench.directional_config(*dims)
    cfg.dt *= 0.5
    return cfg


# words = ceil(nx / 64) * ny * nz
DIMS = [(1, 1, 1), (5, 9, 7), (64, 8, 8), (65, 4, 8), (3, 5, 13), (2, 16, 16), (3, 257, 1), (66, 127, 1),
        (1, 192, 256), (1, 193, 255), (2, 256, 512), (1, 331, 397)]


@pytest.mark.parametrize("solid", [0.0, 0.003, 0.4], ids=["liquid", "few", "many"])
@pytest.mark.parametrize("dims", DIMS, ids=["x".join(map(str, d)) for d in DIMS])
def test_interface_list(dims, solid):
    from mumatscale_amd.lib import Subblock
    cfg = _cfg(*dims)
    nx, ny, nz = dims
    rng = np.random.default_rng(nx + 7 * ny + 31 * nz)
    gr = np.zeros((nz + 2, ny + 2, nx + 2), np.int32)
    gr[1:-1, 1:-1, 1:-1] = rng.random((nz, ny, nx)) < solid
    near = np.zeros(gr.shape, bool)
    for a in range(3):
        for d in (-1, 1):
            near |= np.roll(gr, d, a) > 0            # the halo is liquid, so nothing wraps
    inside = np.zeros(gr.shape, bool)
    inside[1:-1, 1:-1, 1:-1] = True
    want = np.flatnonzero((inside & (gr <= 0) & near).ravel()).astype(np.int32)
    recs = [abi.Grain(), abi.Grain()]
    for q in range(3):
        recs[1].rotmat[q][q] = 1.0
    with Subblock(cfg.params(), cfg.nucleation()) as sb:
        sb.set_grains(recs)
        sb.upload(abi.FIELD_GR, gr)
        for _ in range(2):                           # the counters between launches are left at 0
            assert sb.grow_cell_reduction() == want.size
            assert np.array_equal(sb.interface_list(), want)


# about nx * ny * nz * 1e-18 * density bulk sites
@pytest.mark.parametrize("sites", [40, 256, 300, 700])
def test_nucleation_in_one_launch(sites):
    from mumatscale_amd.lib import Subblock
    cfg = _cfg(24, 23, 25)
    cfg.surf_density = 0.0
    cfg.bulk_density = sites / (24 * 23 * 25 * 1.0e-18)
    cfg.gradient = 0.0
    cfg.velocity = 0.0
    cfg.cool_rate = 2000.0
    cfg.t_init = 933.0
    with Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as a, \
            Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as b:
        born = set()
        for t in range(1, 161):
            a.step(1)
            b.timestep = t
            b.cell_nucleation()
            b.activate_new_grains()
            b.sb_diffuse_alloy_decentered()
            b.fs_change_diffuse()
            b.grow_octahedra()
            b.grow_cell_reduction()
            b.capture_octahedra_diffuse()
            assert a.num_grains == b.num_grains, t
            born.add(a.num_grains)
        assert len(born) > 5
        for f in (abi.FIELD_GR, abi.FIELD_CE, abi.FIELD_CL, abi.FIELD_FS):
            assert np.array_equal(a.download(f).view(np.uint8), b.download(f).view(np.uint8)), f
        for p, q in zip(a.grains(), b.grains()):
            assert bytes(p) == bytes(q)
