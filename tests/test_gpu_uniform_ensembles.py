"""Ensembles in uniform fields: the step count that a solve reports, and that
many particles do not queue for adding to it."""
import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd.device import DeviceEnsemble

pytestmark = pytest.mark.gpu


def ensemble(n, nt, precision, every=0):
    rng = np.random.default_rng(n)
    xv = np.hstack([rng.uniform(-1.0, 1.0, (n, 3)), rng.normal(0.0, 1e5, (n, 3))])
    p = TP.TraceProblem(xv, (0.0, nt * 0.1), (TP.qi / TP.mi, TP.mi, TP.UniformField([1e-4, 0.0, 2e-4]),
                                              TP.UniformField([0.0, 0.0, 1e-8]), TP.ZeroField()))
    return DeviceEnsemble(p, TP.Boris(), xv, dt=0.1, precision=precision,
                          **(dict(savestepinterval=every) if every else dict(save_everystep=False)))


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("n,nt", [(1, 0), (1, 1), (15, 7), (16, 300), (17, 4), (65, 13), (1000, 31)])
def test_particle_steps(precision, n, nt):
    for every in (0, 3):
        e = ensemble(n, nt, precision, every)
        assert [e.run().particle_steps for _ in range(3)] == [n * nt] * 3


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_short_solves_of_many_particles(precision):
    # 20 steps are a fifteenth of 300; with one sum per wave, queueing at one
    # address, they take 0.85 of the time
    ms = [min(e.run().kernel_ms for _ in range(8)) for e in (ensemble(500000, nt, precision) for nt in (20, 300))]
    assert ms[0] < 0.5 * ms[1]
