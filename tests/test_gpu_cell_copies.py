"""A cell copy that a solve built by itself: taken out of use and put back,
with a batch made in between, the results stay those of the same kernels on
the nodes, bit for bit."""
import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd import _lib
from testparticle_amd.device import DeviceBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_batch_survives_dropping_a_copy(precision):
    rng = np.random.default_rng(4)
    L, m, n, nt = 1.0e8, 12, 9001, 100                     # n * nt gathers: the solve builds the copy
    A = rng.normal(0.0, 1e-9, (3, m, m, m)).astype(np.float32 if precision == "fp32c" else np.float64)
    B, on_nodes = [TP.GridField(A, *[np.arange(m) * (L / m)] * 3, bc=TP.PeriodicBC(), layout="nodes",
                                storage="f32" if precision == "fp32c" else "f64") for _ in range(2)]
    xv = np.hstack([rng.uniform(0.0, L, (n, 3)), rng.normal(0.0, 1e6, (n, 3))])
    prob, ref = [TP.TraceProblem(xv, (0.0, nt * 0.3), (TP.qi / TP.mi, TP.mi, TP.ZeroField(), b, TP.ZeroField()))
                 for b in (B, on_nodes)]
    kw = dict(dt=0.3, save_everystep=False, precision=precision)
    ctx = _lib.context(0)
    ctx.check(ctx.L.tpamd_field_grid_cells(ctx.h, on_nodes.handle(ctx), 0))     # none is built from here on
    want = TP.solve(ref, TP.Boris(), **kw)
    auto = TP.solve(prob, TP.Boris(), **kw)
    batch = DeviceBatch([prob, prob], TP.Boris(), **kw)
    h = B.handle(ctx)
    for enable in (0, 1, 0, 0, 1):
        ctx.check(ctx.L.tpamd_field_grid_cells(ctx.h, h, enable))
        batch.run()
        u = batch.u.cpu().numpy().reshape(2 * n, -1, 6)
        for got in (u[:n], u[n:], TP.solve(prob, TP.Boris(), **kw).u_all, auto.u_all):
            np.testing.assert_array_equal(got.view(np.int64), want.u_all.view(np.int64))
    batch.close()
