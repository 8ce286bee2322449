"""Batches on the generic kernels (asked for, or because the instances differ
in wrapping or field kinds) against single solves on the generic kernels, bit
for bit: adaptive ones with particles that stay and leave, and fixed steps."""
import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd import workloads as W

pytestmark = pytest.mark.gpu

L = 1.0e7
TG = 2 * np.pi * TP.mi / (TP.qi * 5e-9)


def problem(n, seed, precision, bc, field="grid"):
    rng = np.random.default_rng(seed)
    m = 8 + seed % 5
    dtype = np.float32 if precision == "fp32c" else np.float64
    if field == "uniform":
        B = TP.UniformField([1e-9, 0.0, 5e-9])
    else:
        def grid(k):
            return TP.GridField(W.turbulent_field(m, L, 5e-9, 0.5, seed + k, dtype=dtype),
                                *W.grid_axes(m, L, periodic=bc == "periodic"),
                                bc={"periodic": TP.PeriodicBC, "clamp": TP.ClampExtrap, "fill": TP.FillExtrap}[bc]())
        B = grid(0) if field == "grid" else TP.LazyTimeInterpolator([0.0, 5 * TG], grid)
    x = rng.uniform(0, L, (n, 3))
    v = W.isotropic_directions(rng, n) * np.sqrt(2 * rng.uniform(1e4, 1e6, n) * TP.qi / TP.mi)[:, None]
    still = rng.random(n) < 0.2
    x[still], v[still] = 0.5 * L, v[still] * 1e-6
    return TP.TraceProblem(np.hstack([x, v]), (0.0, 40 * TG / 25), (TP.qi / TP.mi, TP.mi, TP.ZeroField(), B, TP.ZeroField()))


def bits(s):
    w = np.arange(s.u_all.shape[1]) < s.lengths[:, None]
    return s.lengths, s.retcodes, s.u_all[w].view(np.int64), s.t_all[w].view(np.int64)


def compare(probs, alg, single, batch):
    for pr, g in zip(probs, TP.solve_batch(probs, alg, **batch)):
        if not len(pr.u0):
            assert len(g) == 0
            continue
        for a, b in zip(bits(g), bits(TP.solve(pr, alg, **single))):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("counts", [[1], [7, 8, 9], [55, 56, 57, 63, 64, 65], [0, 127, 0, 128, 129], [3000, 5, 2000]])
@pytest.mark.parametrize("alg,kw", [(TP.AdaptiveBoris(safety=0.1), dict(max_steps=60)), (TP.Boris(), dict(dt=TG / 25))])
def test_generic_kernels_asked_for(precision, counts, alg, kw):
    probs = [problem(n, k, precision, "clamp") for k, n in enumerate(counts)]
    kw = dict(kw, isoutside=TP.OutsideGrid(), save_everystep=False, precision=precision, kernels="generic")
    compare(probs, alg, kw, kw)
    if precision == "fp32c" and len(counts) == 3:
        # these are other kernels than the specialised ones, which round differently
        other = TP.solve_batch(probs, alg, **dict(kw, kernels="auto"))
        assert any((a.u_all != b.u_all).any() for a, b in zip(other, TP.solve_batch(probs, alg, **kw)))


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("alg,kw", [(TP.AdaptiveBoris(safety=0.1), dict(max_steps=60)), (TP.Boris(), dict(dt=TG / 25)),
                                    (TP.MultistepBoris(4, n=3), dict(dt=TG / 25))])
@pytest.mark.parametrize("mix", [("periodic", "clamp", "fill"), ("grid", "uniform", "grid"), ("time", "grid", "time")])
def test_instances_that_differ(precision, mix, alg, kw):
    probs = [problem(n, k, precision, *((m,) if m in ("periodic", "clamp", "fill") else ("clamp", m)))
             for k, (n, m) in enumerate(zip((700, 64, 300), mix))]
    kw = dict(kw, isoutside=TP.OutsideSphere(2 * L), save_everystep=False, precision=precision)
    compare(probs, alg, dict(kw, kernels="generic"), kw)
