"""A call that is rejected leaves nothing behind: no cell copy of its field,
built or on its way, and the next call on another stream gets the same bits as
one on a field that never was in a rejected call."""
import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd import _lib
from testparticle_amd.device import DeviceEnsemble

pytestmark = pytest.mark.gpu

L, M, N, NT = 1.0e8, 96, 9001, 400                # N * NT gathers would build the copy, 170 MB
XV = np.hstack([np.random.default_rng(2).uniform(0.0, L, (N, 3)),
                np.random.default_rng(3).normal(0.0, 1e6, (N, 3))])
KW = dict(dt=0.3, save_everystep=False)


def problem(uxb=False):
    A = np.random.default_rng(1).normal(0.0, 1e-9, (3, M, M, M))
    A[2] += 5e-9
    B = TP.GridField(A, *[np.arange(M) * (L / M)] * 3, bc=TP.PeriodicBC())
    E = TP.UxBField([1e5, 0.0, 0.0], B) if uxb else TP.ZeroField()
    return TP.TraceProblem(XV, (0.0, NT * 0.3), (TP.qi / TP.mi, TP.mi, E, B, TP.ZeroField()))


def rejected_solve(p):
    with pytest.raises(_lib.ArgumentError):
        TP.solve(p, TP.Boris(), workgroup_size=100, **KW)
    with pytest.raises(_lib.ArgumentError):
        TP.solve(p, TP.Boris(), particles_per_lane=7, **KW)


def rejected_device_solve(p):
    e = DeviceEnsemble(p, TP.Boris(), XV, workgroup_size=100, **KW)
    with pytest.raises(_lib.ArgumentError):
        e.run()


def rejected_gradient(p):
    with pytest.raises(_lib.CapacityError):
        TP.loss_gradient(p, dt=0.3, targets=np.zeros((N, 3)), ckpt_interval=2**31 - 1)


@pytest.mark.parametrize("rejected", [rejected_solve, rejected_device_solve, rejected_gradient])
def test_rejected_call_builds_nothing(rejected):
    import torch
    p, ref = problem(), problem()
    ctx = _lib.context(0)
    ctx.check(ctx.L.tpamd_field_grid_cells(ctx.h, ref.p[3].handle(ctx), 0))       # none is built from here on
    want = DeviceEnsemble(ref, TP.Boris(), XV, **KW)
    want.run()
    e = DeviceEnsemble(p, TP.Boris(), XV, **KW)
    rejected(p)                                       # whatever staging it needs is allocated
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    rejected(p)
    assert before - torch.cuda.mem_get_info()[0] < 64 << 20
    built = torch.cuda.mem_get_info()[0]
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        e.run()
    s.synchronize()
    assert built - torch.cuda.mem_get_info()[0] > 128 << 20      # the valid call is the one that builds the copy
    assert torch.equal(e.u.view(torch.int64), want.u.view(torch.int64))
