"""Replay and adjoint step of a Gaussian-beam block, whose growing cells each
evaluate a 400-term quadrature: that their work is spread over the chip.  A
step that writes apart from its inputs does not take much longer than one in
place, and growing cells side by side not much longer than spread ones."""
import ctypes as C

import numpy as np
import pytest
import torch

from mumatscale_amd import abi
from mumatscale_amd.lib import lib

pytestmark = pytest.mark.gpu

DIMS = (128, 96, 64)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _packed(codes):
    nz, ny, nx = codes.shape
    w = (nx + 63) // 64
    c = torch.nn.functional.pad(torch.from_numpy(codes), (0, w * 64 - nx, 1, 1, 1, 1)).reshape(nz + 2, ny + 2, w, 64)
    bit = torch.arange(64, dtype=torch.int64)
    return torch.stack([(((c >> p) & 1) << bit).sum(-1) for p in range(3)], -1).reshape(-1).cuda()


class _Block:
    def __init__(self):
        from mumatscale_amd.workloads import am_track_config
        nx, ny, nz = DIMS
        cfg = am_track_config(*DIMS)
        cfg.cell_size, cfg.dt = 1.0e-6, 1.0e-6
        cfg.laser.update(start=[0.0, ny * 0.5e-6, nz * 1.0e-6])
        self.params = cfg.params(check_negative_ce=False)
        cells = (nx + 2) * (ny + 2) * (nz + 2)
        g = torch.Generator(device="cuda").manual_seed(3)
        rnd = lambda: torch.rand(cells, generator=g, dtype=torch.float64, device="cuda")  # noqa: E731
        self.state = [4.0 + rnd(), 4.0 + rnd(), rnd()]
        self.grads = [rnd() for _ in range(3)]
        self.out = [t.clone() for t in self.grads]
        self.g_param = torch.zeros(3, dtype=torch.float64, device="cuda")
        nb = C.c_int64(0)
        assert lib().mmca_adjoint_workspace_bytes(C.byref(self.params), C.byref(nb)) == abi.OK
        self.ws = torch.zeros((nb.value + 7) // 8, dtype=torch.float64, device="cuda")

    def adjoint(self, codes, out):
        assert lib().mmca_adjoint_step(C.byref(self.params), 300, _ptr(codes), *map(_ptr, self.state),
                                       *map(_ptr, self.grads), *map(_ptr, out), _ptr(self.g_param), _ptr(self.ws),
                                       None) == abi.OK

    def replay(self, codes):
        assert lib().mmca_replay_step(C.byref(self.params), 300, _ptr(codes), *map(_ptr, self.state),
                                      *map(_ptr, self.out), None) == abi.OK


def _ms(f):
    best = 1e9
    for _ in range(4):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        a.record(torch.cuda.default_stream())
        for _ in range(5):
            f()
        b.record(torch.cuda.default_stream())
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) / 5)
    return best


def _codes(planes):
    """Every 16th cell of a row growing in the given planes, the rest solid."""
    nx, ny, nz = DIMS
    c = np.full((nz, ny, nx), abi.BRANCH_SOLID, np.int64)
    c[planes, :, ::16] = abi.BRANCH_GROW
    return _packed(c)


def test_step_apart_against_in_place():
    b = _Block()
    codes = _codes(slice(None, None, 4))
    apart, inplace = _ms(lambda: b.adjoint(codes, b.out)), _ms(lambda: b.adjoint(codes, b.grads))
    assert apart < 2 * inplace, (apart, inplace)


@pytest.mark.parametrize("what", ["replay", "adjoint"])
def test_growing_cells_side_by_side_against_spread(what):
    b = _Block()
    t = {}
    for name, planes in (("spread", slice(None, None, 4)), ("side", slice(48, 64))):
        codes = _codes(planes)
        t[name] = _ms(lambda: b.replay(codes) if what == "replay" else b.adjoint(codes, b.grads))
    assert t["side"] < 2 * t["spread"], t


def test_replay_of_a_recorded_beam_run():
    """Bit for bit the state that the recorded run ended in."""
    from mumatscale_amd import adjoint as ADJ
    from mumatscale_amd.lib import Subblock
    from mumatscale_amd.workloads import am_track_config, voronoi_substrate
    cfg = am_track_config(70, 37, 21)
    cfg.cell_size, cfg.dt = 1.0e-6, 2.0e-6
    cfg.laser.update(power=60.0, spot=130e-6, sub_init_temp=600.0, start=[0.0, 18.5e-6, 21e-6])
    gr, recs = voronoi_substrate(cfg, 40, 5)
    fs = np.zeros(gr.shape)
    fs[1:-1, 1:-1, 1:-1] = 1.0
    with Subblock(cfg.params(check_negative_ce=False), cfg.nucleation()) as sb:
        sb.set_grains(recs)
        sb.upload(abi.FIELD_GR, gr)
        sb.upload(abi.FIELD_FS, fs)
        traj = ADJ.record(sb, 120)
        want = [sb.download(f).reshape(-1) for f in (abi.FIELD_CE, abi.FIELD_CL, abi.FIELD_FS)]
    assert (want[2].reshape(gr.shape)[1:-1, 1:-1, 1:-1] < 1.0).any()
    got, _ = ADJ.replay(traj, cfg.d_liq, cfg.d_sol, cfg.part_coef)
    for w, t in zip(want, got):
        assert np.array_equal(t.cpu().numpy().view(np.uint64), w.view(np.uint64))
