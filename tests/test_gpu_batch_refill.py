"""Adaptive batches where a wave's refills change: chunks around the lanes and
the refill threshold, fewer chunks than slices, many instances, lanes held by
particles that never leave; against single solves, bit for bit."""
import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd import workloads as W

pytestmark = pytest.mark.gpu

L = 1.0e7
TG = 2 * np.pi * TP.mi / (TP.qi * 5e-9)


def problem(n, trapped, seed, precision, generic):
    rng = np.random.default_rng(seed)
    m = 8 + seed % 5
    A = W.turbulent_field(m, L, 5e-9, 0.5, seed, dtype=np.float32 if precision == "fp32c" else np.float64)
    B = TP.GridField(A, *W.grid_axes(m, L, periodic=False), bc=TP.FillExtrap() if generic and seed % 2 else TP.ClampExtrap())
    x = rng.uniform(0, L, (n, 3))
    v = W.isotropic_directions(rng, n) * np.sqrt(2 * rng.uniform(1e4, 1e6, n) * TP.qi / TP.mi)[:, None]
    still = rng.random(n) < trapped
    x[still], v[still] = 0.5 * L, v[still] * 1e-6
    return TP.TraceProblem(np.hstack([x, v]), (0.0, 1e6 * TG), (TP.qi / TP.mi, TP.mi, TP.ZeroField(), B, TP.ZeroField()))


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("counts,trapped,generic", [([1], 0.0, False), ([7, 8, 9], 0.5, False), ([55, 56, 57, 63, 64, 65], 0.1, False),
                                                    ([0, 127, 0, 128, 129], 0.2, False), ([1] * 70, 0.3, False),
                                                    ([3000, 5, 2000], 0.15, False), ([3000, 5, 2000], 1.0, False),
                                                    ([700, 64, 300], 0.2, True), ([300000, 17], 0.0, False)])
def test_batch_refills_match_single_solves(precision, counts, trapped, generic):
    probs = [problem(n, trapped, k, precision, generic) for k, n in enumerate(counts)]
    kw = dict(isoutside=TP.OutsideGrid(), max_steps=60, save_everystep=False, precision=precision)
    alg = TP.AdaptiveBoris(safety=0.1)
    sols = TP.solve_batch(probs, alg, **kw)
    for pr, g in zip(probs, sols):
        if not len(pr.u0):
            assert len(g) == 0
            continue
        s = TP.solve(pr, alg, **kw)
        np.testing.assert_array_equal(g.retcodes, s.retcodes)
        np.testing.assert_array_equal(g.lengths, s.lengths)
        written = np.arange(g.u_all.shape[1]) < g.lengths[:, None]
        np.testing.assert_array_equal(g.u_all[written].view(np.int64), s.u_all[written].view(np.int64))
        np.testing.assert_array_equal(g.t_all[written].view(np.int64), s.t_all[written].view(np.int64))
