"""The uniform-field and dipole kernels at the step counts and save intervals
where their loops end (steps in threes and in twos, remainders, saves at every
step), against the generic kernels, bit for bit with the signs of zeros."""
import numpy as np
import pytest

import testparticle_amd as TP

pytestmark = pytest.mark.gpu


def assert_same_bits(prob, precision, **kw):
    a = TP.solve(prob, TP.Boris(), precision=precision, **kw)
    b = TP.solve(prob, TP.Boris(), precision=precision, kernels="generic", **kw)
    np.testing.assert_array_equal(a.lengths, b.lengths)
    np.testing.assert_array_equal(a.retcodes, b.retcodes)
    for i in range(len(a)):
        n = a.lengths[i]
        np.testing.assert_array_equal(a.u_all[i, :n].view(np.int64), b.u_all[i, :n].view(np.int64))
        np.testing.assert_array_equal(a.t_all[i, :n].view(np.int64), b.t_all[i, :n].view(np.int64))
    return a


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("every", [1, 2, 3, 4, 5, 10])
def test_uniform_fields_at_every_remainder(precision, every):
    rng = np.random.default_rng(every)
    xv = rng.normal(0.0, 1.0, (67, 6)) * [1, 1, 1, 1e5, 1e5, 1e5]
    xv[::5, 2] = -0.0
    xv[::5, 5] = -0.0
    q2m, dt = TP.qi / TP.mi, 0.1
    B = TP.UniformField([2e-9, 0.0, 1e-8])
    for E in (TP.ZeroField(), TP.UniformField([-0.0, -0.0, -0.0]), TP.UniformField([0.0, -0.0, 0.0]),
              TP.UniformField([1e-4, 0.0, -2e-4])):
        for sign in (1.0, -1.0):
            for nt in (0, 1, 2, 3, 4, 5, 6, 7, 13, 31):
                prob = TP.TraceProblem(xv, (0.0, nt * dt), (sign * q2m, TP.mi, E, B, TP.ZeroField()))
                kw = dict(dt=dt, savestepinterval=every, save_start=nt % 2 == 0, save_end=nt % 3 == 0)
                assert_same_bits(prob, precision, **kw)
                assert_same_bits(prob, precision, **dict(kw, save_everystep=False))


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("every", [1, 2, 3, 7])
def test_dipole_at_every_remainder(precision, every):
    rng = np.random.default_rng(10 + every)
    n = 67
    r = rng.uniform(2.0, 7.0, n) * TP.Re
    ph = rng.uniform(0.0, 2 * np.pi, n)
    xv = np.stack([r * np.cos(ph), r * np.sin(ph), rng.uniform(-1.0, 1.0, n) * TP.Re, *rng.normal(0.0, 2e7, (3, n))], 1)
    xv[::5, 2] = 0.0                  # the equator: two components of B are zero
    xv[1::5, 5] = -0.0
    xv[2::7, 3:] = 0.0                # at rest
    dts = 2 * np.pi * TP.mi / (TP.qi * 3.12e-5 * (TP.Re / r) ** 3) / 32
    dip = TP.DipoleField(3.12e-5, TP.Re)
    left = 0
    for q in (1.0, -1.0):
        for nt in (1, 2, 3, 4, 9, 60):
            prob = TP.TraceProblem(xv, (0.0, 0.0), (q * TP.qi / TP.mi, TP.mi, TP.ZeroField(), dip, TP.ZeroField()))
            for out in (None, TP.InsideSphere(2.5 * TP.Re) | TP.OutsideSphere(6.5 * TP.Re),
                        TP.InsideSphere(2.5 * TP.Re) | TP.OutsideBox([-6 * TP.Re] * 3, [6 * TP.Re] * 3)):
                for kw in (dict(savestepinterval=every), dict(save_everystep=False), dict(save_start=False)):
                    a = assert_same_bits(prob, precision, dts=dts, nsteps=nt, isoutside=out, **kw)
                    left += int((a.retcodes == 1).sum())
    assert left > 100
