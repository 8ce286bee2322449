"""The dipole kernel's own division and square root, and particles whose field
has components that are exactly zero at every step."""
import json
import os
import subprocess

import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd.device import DeviceEnsemble

pytestmark = pytest.mark.gpu


def test_division_and_root_across_their_ranges():
    # random operands over the whole ranges that the kernel uses them in, the
    # edges and the pairs that it forms among them: not one bit may differ
    exe = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "testparticle.jl_amd",
                       "_build", "shared_div_check")
    r = subprocess.run([exe, "2048"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    out = json.loads(r.stdout)
    for n, bad in (("pairs", "differing"), ("roots", "roots_differing")):
        assert out[n] >= 1e9 and out[bad] == 0


def population(rng, n, kind):
    """Protons on the equator, moving in it (one component of v -0.0 for some),
    or on the axis, moving along it; "z": anywhere, moving in any direction."""
    r = rng.uniform(3.0, 7.0, n) * TP.Re
    ph, sp = rng.uniform(0.0, 2 * np.pi, (2, n))
    v = rng.uniform(1e6, 3e7, n)
    zero = np.where(np.arange(n) % 2, 0.0, -0.0)
    if kind == "equator":
        xv = np.stack([r * np.cos(ph), r * np.sin(ph), zero, v * np.cos(sp), v * np.sin(sp), -zero], 1)
        xv[::7, :2] = np.stack([r[::7], zero[::7]], 1)            # on the x axis
    elif kind == "axis":
        up = np.where(np.arange(n) % 3, 1.0, -1.0)
        xv = np.stack([zero, -zero, r * up, -zero, zero, v * up], 1)
    else:
        xv = np.stack([r * np.cos(ph), r * np.sin(ph), zero, v * np.cos(sp), v * np.sin(sp) * 0.6, v * np.sin(sp) * 0.8], 1)
    return xv, 2 * np.pi * TP.mi / (TP.qi * 3.12e-5 * (TP.Re / r) ** 3) / 32


def problem(xv, sign=1.0, scale=1.0):
    return TP.TraceProblem(xv, (0.0, 0.0), (sign * TP.qi / TP.mi, TP.mi, TP.ZeroField(),
                                            TP.DipoleField(3.12e-5 * scale, TP.Re), TP.ZeroField()))


# scales of the field: the belt's, one where |h k| is below what the zeros'
# shortcut asks for, and the edges of the kernel's range
@pytest.mark.parametrize("kind", ["equator", "axis"])
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("scale", [1.0, -1.0, 1e-39, 1e-100, 1e12])
def test_zero_components_bit_for_bit(kind, sign, scale):
    xv, dts = population(np.random.default_rng(6), 67, kind)
    for out in (None, TP.InsideSphere(2.9 * TP.Re) | TP.OutsideSphere(7.2 * TP.Re),
                TP.InsideSphere(2.9 * TP.Re) | TP.OutsideBox([-6 * TP.Re] * 3, [6 * TP.Re] * 3)):
        kw = dict(dts=dts, nsteps=150, savestepinterval=3, isoutside=out)
        a = TP.solve(problem(xv, sign, scale), TP.Boris(), **kw)
        b = TP.solve(problem(xv, sign, scale), TP.Boris(), kernels="generic", **kw)
        np.testing.assert_array_equal(a.lengths, b.lengths)
        np.testing.assert_array_equal(a.retcodes, b.retcodes)
        w = np.arange(a.u_all.shape[1]) < a.lengths[:, None]
        np.testing.assert_array_equal(a.u_all[w].view(np.int64), b.u_all[w].view(np.int64))
        np.testing.assert_array_equal(a.t_all[w].view(np.int64), b.t_all[w].view(np.int64))


def test_equator_is_not_slower_than_the_rest():
    # a step that is thrown away and formed again by the generic arithmetic
    # takes 2.4 times as long; the way around it is some 10 instructions of 110
    ms = {}
    for kind in ("equator", "z"):
        xv, dts = population(np.random.default_rng(8), 262144, kind)
        e = DeviceEnsemble(problem(xv), TP.Boris(), xv, dts=dts, nsteps=500, save_everystep=False,
                           isoutside=TP.InsideSphere(TP.Re))
        ms[kind] = min(e.run().kernel_ms for _ in range(8))
    assert ms["equator"] < 1.3 * ms["z"]
