"""Solves that gather from two grids a step (gridded E and B, or snapshots
blended in time), and the generic kernels reading the cell-replicated copy:
the same bits as the generic kernels on the node arrays, and in FP64 as the
oracle."""
import numpy as np
import pytest

import testparticle_amd as TP
from parity import assert_bitwise, run_oracle

pytestmark = pytest.mark.gpu

L, Q2M = 1.0e8, TP.qi / TP.mi
SHAPE = (7, 9, 6)
BCS = {"periodic": TP.PeriodicBC, "clamp": TP.ClampExtrap, "fill": TP.FillExtrap}


def axes(bc):
    return [np.arange(n) * (L / n if bc == "periodic" else L / (n - 1)) for n in SHAPE]


def nodes(rng, scale, mean, dtype):
    return (rng.normal(0.0, scale, (3,) + SHAPE) + np.array(mean)[:, None, None, None]).astype(dtype)


def particles(rng, n):
    return np.hstack([rng.uniform(0.2 * L, 0.8 * L, (n, 3)), rng.normal(0.0, 1.5e6, (n, 3))])


def problem(xv, nt, E, B):
    return TP.TraceProblem(xv, (0.0, nt * 0.3), (Q2M, TP.mi, E, B, TP.ZeroField()))


def same(a, b):
    np.testing.assert_array_equal(a.lengths, b.lengths)
    np.testing.assert_array_equal(a.retcodes, b.retcodes)
    for i in range(len(a)):
        n = a.lengths[i]
        np.testing.assert_array_equal(a.u_all[i, :n], b.u_all[i, :n])
        np.testing.assert_array_equal(a.t_all[i, :n], b.t_all[i, :n])


def eb(rng, bc, dtype, layout):
    ax = axes(bc)
    rs = np.random.default_rng(rng)
    f = [TP.GridField(nodes(rs, s, m, dtype), *ax, bc=BCS[bc](), layout=layout)
         for s, m in ((1e-3, (0.0, 5e-4, 0.0)), (2e-9, (0.0, 0.0, 5e-9)))]
    return f


@pytest.mark.parametrize("bc", list(BCS))
@pytest.mark.parametrize("precision,dtype", [("fp64", np.float64), ("fp64", np.float32), ("fp32c", np.float32)])
@pytest.mark.parametrize("n,nt", [(1, 1), (63, 40), (65, 200), (300, 333)])
def test_gridded_e_and_b(precision, dtype, bc, n, nt):
    xv = particles(np.random.default_rng(n), n)
    out = None if bc == "periodic" else TP.OutsideGrid()
    for kw in (dict(savestepinterval=7), dict(save_everystep=False)):
        kw.update(dt=0.3, precision=precision, isoutside=out)
        p = problem(xv, nt, *eb(n, bc, dtype, "cells"))
        a = TP.solve(p, TP.Boris(), **kw)
        same(a, TP.solve(problem(xv, nt, *eb(n, bc, dtype, "nodes")), TP.Boris(), kernels="generic", **kw))
        if precision == "fp64" and nt < 300:
            kw.pop("precision")
            assert_bitwise(a, run_oracle(p, TP.Boris(), **kw))


@pytest.mark.parametrize("bc", list(BCS))
@pytest.mark.parametrize("precision,dtype", [("fp64", np.float64), ("fp64", np.float32), ("fp32c", np.float32)])
@pytest.mark.parametrize("snaps", [1, 2, 5])
def test_snapshots(precision, dtype, bc, snaps):
    rng = np.random.default_rng(snaps)
    n, nt = 4200, 200                 # enough gathers for the solve to build the cells
    ax = axes(bc)
    data = [nodes(rng, 2e-9, (0.0, 0.0, 5e-9), dtype) for _ in range(snaps)]
    xv = particles(rng, n)
    out = None if bc == "periodic" else TP.OutsideGrid()
    times = np.linspace(0.1, 0.8, snaps) * nt * 0.3 if snaps > 1 else [5.0]

    def fields(uxb):
        B = TP.LazyTimeInterpolator(times, lambda i: TP.GridField(data[i - 1], *ax, bc=BCS[bc]()))
        return (TP.UxBField([3e5, 0.0, -1e5], B) if uxb else TP.UniformField([0.0, 5e-4, 0.0])), B

    for uxb in (False, True):
        kw = dict(dt=0.3, precision=precision, isoutside=out, savestepinterval=60)
        p = problem(xv, nt, *fields(uxb))
        a = TP.solve(p, TP.Boris(), **kw)
        b = TP.solve(problem(xv, nt, *fields(uxb)), TP.Boris(), kernels="generic", **kw)
        same(a, b)
        # the generic kernels on the copy that the first solve built
        same(TP.solve(p, TP.Boris(), kernels="generic", **kw), b)
        m = TP.solve(p, TP.MultistepBoris(4, n=3), **kw)
        same(m, TP.solve(problem(xv, nt, *fields(uxb)), TP.MultistepBoris(4, n=3), kernels="generic", **kw))


@pytest.mark.parametrize("bc", list(BCS))
@pytest.mark.parametrize("precision,dtype", [("fp64", np.float64), ("fp32c", np.float32)])
def test_generic_kernels_read_the_cells(precision, dtype, bc):
    xv = particles(np.random.default_rng(9), 130)
    out = None if bc == "periodic" else TP.OutsideGrid()
    c, g = problem(xv, 60, *eb(3, bc, dtype, "cells")), problem(xv, 60, *eb(3, bc, dtype, "nodes"))
    kw = dict(precision=precision, isoutside=out)
    for alg, k in ((TP.Boris(), dict(dt=0.3, save_fields=True, save_work=True, savestepinterval=9)),
                   (TP.MultistepBoris(6, n=2), dict(dt=0.3, savestepinterval=9)),
                   (TP.AdaptiveBoris(0.1), dict(max_steps=50, savestepinterval=5))):
        same(TP.solve(c, alg, **kw, **k), TP.solve(g, alg, kernels="generic", **kw, **k))
    x = np.random.default_rng(1).uniform(-0.2 * L, 1.2 * L, (500, 3))
    np.testing.assert_array_equal(c.p[3](x, precision=precision), g.p[3](x, precision=precision))
