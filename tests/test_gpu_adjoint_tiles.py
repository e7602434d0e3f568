"""The one-pass adjoint step (outputs apart from the inputs) at the edges of
its tiles of 64 x 8 cells and of its walks, against the two-pass step that
updates the incoming derivatives in place: the fields bit for bit, twice with
one workspace, halo cells left alone; and the parameter derivatives, which the
two sum in different orders, within n eps sum|terms| of each other for liquid
and solid cells (the terms formed with torch)."""
import ctypes as C

import numpy as np
import pytest
import torch

from mumatscale_amd import abi
from mumatscale_amd.lib import lib
from mumatscale_amd.workloads import seeded_grains_config

pytestmark = pytest.mark.gpu

DIMS = [(1, 1, 1), (63, 7, 5), (64, 8, 6), (65, 9, 7), (2, 17, 33), (129, 1, 4), (70, 25, 130)]


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _packed(codes, nx):
    nz, ny, _ = codes.shape
    w = (nx + 63) // 64
    full = np.zeros((nz + 2, ny + 2, w * 64), np.uint64)
    full[1:-1, 1:-1, :nx] = codes
    bit = np.arange(64, dtype=np.uint64)
    words = [(((full >> np.uint64(p)) & np.uint64(1)).reshape(nz + 2, ny + 2, w, 64) << bit).sum(-1, dtype=np.uint64)
             for p in range(3)]
    return torch.from_numpy(np.stack(words, -1).reshape(-1).view(np.uint8).copy()).cuda()


def _step(params, codes, state, grads, out, ws):
    g_param = torch.zeros(3, dtype=torch.float64, device="cuda")
    assert lib().mmca_adjoint_step(C.byref(params), 5, _ptr(codes), *(_ptr(t) for t in state),
                                   *(_ptr(t) for t in grads), *(_ptr(t) for t in out), _ptr(g_param), _ptr(ws),
                                   None) == abi.OK
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in out], g_param.cpu().numpy()


@pytest.mark.parametrize("wall", [1, 0], ids=["walls", "open"])
@pytest.mark.parametrize("dims", DIMS, ids=["x".join(map(str, d)) for d in DIMS])
def test_one_pass_matches_two(dims, wall):
    nx, ny, nz = dims
    cfg = seeded_grains_config(n=128, nseeds=1, seed=4)
    cfg.sbdim = [nx, ny, nz]
    cfg.fixed = []
    cfg.pad_bndy = [wall] * 3
    params = cfg.params(check_negative_ce=False)
    rng = np.random.default_rng(nx + 3 * ny + 11 * nz + wall)
    shape = (nz + 2, ny + 2, nx + 2)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    nb = C.c_int64(0)
    assert lib().mmca_adjoint_workspace_bytes(C.byref(params), C.byref(nb)) == abi.OK
    ws = torch.zeros((nb.value + 7) // 8, dtype=torch.float64, device="cuda")
    for top in (5, 2):                               # all branches; liquid and solid
        codes = rng.integers(0, top, size=(nz, ny, nx))
        packed = _packed(codes, nx)
        h = [1.0 + 9.0 * rng.random(shape), 1.0 + 9.0 * rng.random(shape), rng.random(shape)]
        gh = [rng.normal(size=shape) for _ in range(3)]
        state, grads = [dev(a) for a in h], [dev(a) for a in gh]
        one, p1 = _step(params, packed, state, grads, [torch.full_like(t, 7.0) for t in grads], ws)
        inpl = [t.clone() for t in grads]
        two, p2 = _step(params, packed, state, inpl, inpl, ws)
        inner = (slice(1, -1),) * 3
        for a, b in zip(one, two):
            assert np.array_equal(a[inner].view(np.int64), b[inner].view(np.int64))
            a[inner] = 7.0
            assert np.all(a == 7.0)
        if top == 5:
            continue
        # sums of |terms|, from the formulas of the branches and the stencil
        ce, cl, fs = h
        solid = codes == abi.BRANCH_SOLID
        dtx = params.dt / params.cell_size ** 2
        kinv = 1.0 / params.part_coef
        ga, gb = gh[0][inner], gh[1][inner]
        lam = ga + gb * np.where(solid, kinv, 1.0)
        cen = ce[inner].copy()
        s_f = np.zeros(codes.shape)
        s_1 = np.zeros(codes.shape)
        for ax in (2, 1, 0):
            for d in (1, -1):
                sl = [slice(1, -1)] * 3
                sl[ax] = slice(2, None) if d == 1 else slice(0, -2)
                f = 0.5 * (fs[inner] + fs[tuple(sl)])
                dc = np.abs(cl[tuple(sl)] - cl[inner])
                s_f += np.abs(lam) * f * dc * dtx
                s_1 += np.abs(lam) * dc * dtx
                cen += (params.d_sol * f + params.d_liq * (1 - f)) * dtx * dc
        bound = np.array([s_1.sum(), s_f.sum(), (np.abs(gb) * cen * kinv * kinv * solid).sum()])
        n = 8 * codes.size + 64                      # terms and roundings of each
        assert np.all(np.abs(p1 - p2) <= n * 2.0 ** -52 * bound), (p1, p2, bound)
        assert solid.any() == (p1[2] != 0.0)
