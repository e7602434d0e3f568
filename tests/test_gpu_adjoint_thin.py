"""The adjoint step of boxes one or two planes or rows thin: apart from its
inputs it does not take longer than in place, and gives the same bits."""
import ctypes as C

import pytest
import torch

from mumatscale_amd import abi
from mumatscale_amd.lib import lib
from mumatscale_amd.workloads import seeded_grains_config

pytestmark = pytest.mark.gpu


def _ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("dims", [(1000, 1000, 1), (1000, 900, 2), (300, 1, 300), (300, 300, 1), (65, 2, 130)],
                         ids=lambda d: "x".join(map(str, d)))
def test_apart_against_in_place(dims):
    nx, ny, nz = dims
    cfg = seeded_grains_config(n=128, nseeds=1)
    cfg.sbdim = list(dims)
    cfg.fixed = []
    params = cfg.params(check_negative_ce=False)
    cells = (nx + 2) * (ny + 2) * (nz + 2)
    g = torch.Generator(device="cuda").manual_seed(nx + ny + nz)
    rnd = lambda: torch.rand(cells, generator=g, dtype=torch.float64, device="cuda")  # noqa: E731
    state, grads = [1.0 + rnd(), 1.0 + rnd(), rnd()], [rnd() for _ in range(3)]
    nb = C.c_int64(0)
    assert lib().mmca_adjoint_workspace_bytes(C.byref(params), C.byref(nb)) == abi.OK
    ws = torch.zeros((nb.value + 7) // 8, dtype=torch.float64, device="cuda")
    assert lib().mmca_record_bytes(C.byref(params), C.byref(nb)) == abi.OK
    # liquid and solid cells
    words = torch.randint(-2 ** 62, 2 ** 62, (nb.value // 24, 3), generator=g, device="cuda", dtype=torch.int64)
    words[:, 1:] = 0
    codes = words.reshape(-1)
    g_param = torch.zeros(3, dtype=torch.float64, device="cuda")

    def step(out):
        assert lib().mmca_adjoint_step(C.byref(params), 5, _ptr(codes), *map(_ptr, state), *map(_ptr, grads),
                                       *map(_ptr, out), _ptr(g_param), _ptr(ws), None) == abi.OK

    apart = [torch.zeros_like(t) for t in grads]
    step(apart)
    keep = [t.clone() for t in grads]
    step(grads)
    torch.cuda.synchronize()
    for a, b in zip(apart, grads):
        inner = (slice(1, -1),) * 3
        shape = (nz + 2, ny + 2, nx + 2)
        assert torch.equal(a.reshape(shape)[inner], b.reshape(shape)[inner])

    def ms(out):
        best = 1e9
        for _ in range(6):
            for t, k in zip(grads, keep):
                t.copy_(k)
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            a.record(torch.cuda.default_stream())
            for _ in range(50):
                step(out)
            b.record(torch.cuda.default_stream())
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) / 50)
        return best

    t = ms(apart), ms(grads)
    assert t[0] < 1.4 * t[1], t
