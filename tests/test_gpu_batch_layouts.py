"""A batch's results do not depend on the solves that ran before it: one of
its fields may have got a cell copy from a solve meanwhile, on all entry
points and beside a field whose copy was asked for."""
import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd.device import DeviceBatch, solve_batch_noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layouts", [("nodes", "nodes"), ("nodes", "cells"), ("cells", "nodes")])
@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_batch_after_a_solve_of_one_field(precision, layouts):
    rng = np.random.default_rng(11)
    L, m, n, nt = 1.0e8, 14, 70001, 100              # n * nt gathers: a solve builds a copy
    dtype = np.float32 if precision == "fp32c" else np.float64
    q2m = TP.qi / TP.mi

    def probs():
        out = []
        for k, layout in enumerate(layouts):
            A = np.random.default_rng(k).normal(0.0, 1e-9, (3, m, m + k, m)).astype(dtype)
            A[2] += 5e-9
            B = TP.GridField(A, *[np.arange(s) * (L / s) for s in A.shape[1:]], bc=TP.PeriodicBC(), layout=layout)
            out.append(TP.TraceProblem(xv, (0.0, nt * 0.3), (q2m, TP.mi, TP.ZeroField(), B, TP.ZeroField())))
        return out

    xv = np.hstack([rng.uniform(0.0, L, (n, 3)), rng.normal(0.0, 1e6, (n, 3))])
    kw = dict(dt=0.3, save_everystep=False, precision=precision)

    def written(sols):
        return np.concatenate([s.u_all[np.arange(s.u_all.shape[1]) < s.lengths[:, None]] for s in sols])

    def results(ps):
        dev = DeviceBatch(ps, TP.Boris(), **kw)
        dev.run()
        u = [dev.u.cpu().numpy()]
        dev.close()
        u.append(written(TP.solve_batch(ps, TP.Boris(), **kw)))
        small = [TP.TraceProblem(xv[:700], p.tspan, p.p) for p in ps]
        u.append(solve_batch_noalloc(small, TP.Boris(), **kw)[0].cpu().numpy())
        u.append(written(TP.solve_batch(small, TP.AdaptiveBoris(0.1), precision=precision, save_everystep=False,
                                        max_steps=40)))
        return [a.reshape(-1).view(np.int64) for a in u]

    ps = probs()
    want = results(ps)
    for solved in (0, 1):
        TP.solve(ps[solved], TP.Boris(), **kw)
        for got, w in zip(results(ps), want):
            np.testing.assert_array_equal(got, w)
