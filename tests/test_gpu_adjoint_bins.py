"""The bin sums of the grid gradient (bins split over workgroups, cells summed
by a whole workgroup) against the sorted path, which a grid of more than
2,048 bins takes: the same field embedded in such a grid.  That holds while no
particle reaches the small grid's upper faces, past which it is clamped."""
import numpy as np
import pytest

import testparticle_amd as TP

pytestmark = pytest.mark.gpu

H = 65536.0                            # a power of two: both grids locate alike
SMALL, LARGE = (26, 24, 22), (110, 105, 95)


def population(where, n, nsteps):
    rng = np.random.default_rng(n + nsteps)
    A = rng.normal(0.0, 1e-8, (3,) + LARGE).astype(np.float32)
    x = rng.uniform(6.0, 16.0, (n, 3))
    v = rng.normal(0.0, 1e5, (n, 3))
    if where == "point":
        x, v = 12.5 + rng.uniform(-0.1, 0.1, (n, 3)), v * 1e-4
    elif where == "line":
        x[:, 1:], v = 12.5, v * 1e-4
    elif where == "slow spread":
        v *= 0.1
    xv = np.concatenate([x * H, v], 1)
    tg = x * H + rng.normal(0.0, H, (n, 3))
    return A, xv, tg


def gradient(A, shape, xv, tg, nsteps, precision):
    a = np.ascontiguousarray(A[:, :shape[0], :shape[1], :shape[2]])
    B = TP.GridField(a, *[np.arange(m) * H for m in shape], bc=TP.ClampExtrap(),
                     storage="f32" if precision == "fp32c" else "f64")
    prob = TP.TraceProblem(xv, (0.0, nsteps * 0.05), (TP.qi / TP.mi, TP.mi, TP.ZeroField(), B, TP.ZeroField()))
    return TP.loss_gradient(prob, dt=0.05, targets=tg, precision=precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
@pytest.mark.parametrize("where,n,nsteps", [("spread", 1, 1), ("spread", 257, 9), ("point", 33, 1), ("point", 65, 3),
                                            ("point", 20011, 40), ("line", 5003, 64), ("slow spread", 20011, 40)])
def test_bins_against_the_sorted_path(precision, where, n, nsteps):
    A, xv, tg = population(where, n, nsteps)
    reach = np.linalg.norm(xv[:, 3:], axis=1) * (nsteps * 0.05) / H        # B does no work
    assert (xv[:, :3] / H + reach[:, None] < np.array(SMALL) - 1).all()
    a = gradient(A, SMALL, xv, tg, nsteps, precision)
    b = gradient(A, LARGE, xv, tg, nsteps, precision)
    assert a.loss == pytest.approx(b.loss, rel=1e-12)
    np.testing.assert_array_equal(a.dL_dxv0, b.dL_dxv0)
    # the same terms summed in double in another order
    scale = np.abs(b.dL_dB).max()
    assert scale > 0 and np.isfinite(scale)
    inner = b.dL_dB[:, :SMALL[0], :SMALL[1], :SMALL[2]]
    np.testing.assert_allclose(a.dL_dB, inner, rtol=0, atol=1e-10 * scale)
    assert np.count_nonzero(b.dL_dB) == np.count_nonzero(inner)

