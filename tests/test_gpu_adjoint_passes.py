"""The reverse sweep's passes at the sizes where they end: particle counts
around a block, step counts around a pass, the whole trajectory against
checkpoints, both layouts of the grid gradient."""
import ctypes as C

import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd import _lib
from testparticle_amd import workloads as W
from testparticle_amd.solve import make_desc

pytestmark = pytest.mark.gpu


def gradient(B, xv0, dt, nsteps, tg, precision, interval, flags):
    prob = TP.TraceProblem(xv0, (0.0, nsteps * dt), (TP.qi / TP.mi, TP.mi, TP.ZeroField(), B, TP.ZeroField()))
    d = make_desc(prob, TP.Boris(), dt=dt, precision=precision, save_everystep=False)
    d.flags |= flags
    ctx = _lib.context(0)
    hB = B.handle(ctx)
    n = len(xv0)
    loss, gB, gx, st = np.zeros(1), np.full(B.data.size, np.nan), np.full((n, 6), np.nan), _lib.Stats()
    with ctx.lock:
        ctx.check(ctx.L.tpamd_adjoint(ctx.h, C.byref(d), hB, _lib.dptr(xv0), n, _lib.dptr(tg), interval,
                                      _lib.dptr(loss), _lib.dptr(gB), _lib.dptr(gx), C.byref(st)), st)
    nx, ny, nz = B.shape
    gB = gB.reshape(3, nx, ny, nz) if flags & _lib.FLAG_GRADIENT_BY_COMPONENT \
        else gB.reshape(nz, ny, nx, 3).transpose(3, 2, 1, 0)
    return loss[0], gB, gx


@pytest.mark.parametrize("bc", ["periodic", "clamp"])
@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("n,nsteps,interval", [(1, 1, 1), (63, 7, 3), (256, 8, 8), (257, 15, 4), (255, 16, 16),
                                               (300, 33, 64), (513, 40, 9)])
def test_whole_trajectory_against_checkpoints(precision, bc, n, nsteps, interval):
    w, A = W.turbulent_box(N=n, n=20, nsteps=nsteps, dtype=np.float32)
    shape = (20, 17, 13)
    A = np.ascontiguousarray(A[:, :shape[0], :shape[1], :shape[2]])
    L = w.extra["L"]
    ax = [np.arange(m) * (L / m) for m in shape]
    tg = np.random.default_rng(n).uniform(0.0, L, (n, 3))
    storage = "f32" if precision == "fp32c" else "f64"
    got = []
    for layout in ("cells", "nodes"):
        B = TP.GridField(A, *ax, bc=TP.PeriodicBC() if bc == "periodic" else TP.ClampExtrap(), storage=storage,
                         layout=layout)
        for flags in (0, _lib.FLAG_GRADIENT_BY_COMPONENT, _lib.FLAG_CHECKPOINTS):
            got.append(gradient(B, w.xv0, w.dt, nsteps, tg, precision, interval, flags))
    # per particle the arithmetic is the same; the grid gradient sums the same
    # terms in double in another order: some 1e5 of them, of one sign or not
    scale = np.abs(got[0][1]).max()
    assert scale > 0 and np.isfinite(scale)
    for loss, gB, gx in got[1:]:
        assert loss == pytest.approx(got[0][0], rel=1e-12)
        np.testing.assert_array_equal(gx, got[0][2])
        np.testing.assert_allclose(gB, got[0][1], rtol=0, atol=1e-10 * scale)
