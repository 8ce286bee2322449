"""The adjoint's workspace: where one allocation of the whole trajectory
cannot be had, the call falls back on checkpoints; checkpoints on request,
at every interval."""
import os
import subprocess
import sys

import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd import workloads as W

pytestmark = pytest.mark.gpu


def case(n, nsteps, precision):
    w, A = W.turbulent_box(N=n, n=20, nsteps=nsteps, dtype=np.float32 if precision == "fp32c" else np.float64)
    B = TP.GridField(A, *W.grid_axes(20, w.extra["L"]), bc=TP.PeriodicBC())
    p = TP.TraceProblem(w.xv0, (0.0, nsteps * w.dt), (TP.qi / TP.mi, TP.mi, TP.ZeroField(), B, TP.ZeroField()))
    # close targets: the loss and its gradients stay within the double range
    return p, dict(dt=w.dt, targets=w.xv0[:, :3], precision=precision)


@pytest.mark.parametrize("precision", ["fp64", "fp32c"])
def test_checkpoints_at_every_interval(precision):
    p, kw = case(513, 100, precision)
    whole = TP.loss_gradient(p, **kw)
    scale = np.abs(whole.dL_dB).max()
    for k in (1, 7, 32, 99, 100, 1000):
        r = TP.loss_gradient(p, ckpt_interval=k, checkpoints=True, **kw)
        assert r.loss == pytest.approx(whole.loss, rel=1e-12)
        np.testing.assert_array_equal(r.dL_dxv0, whole.dL_dxv0)
        np.testing.assert_allclose(r.dL_dB, whole.dL_dB, rtol=0, atol=1e-10 * scale)


def limited(n, nsteps):
    """In a process of its own whose single allocations are limited."""
    import torch
    try:
        torch.empty(4 << 30, dtype=torch.uint8, device="cuda")
        print("no limit")
        return
    except torch.OutOfMemoryError:
        pass
    p, kw = case(n, nsteps, "fp32c")
    a = TP.loss_gradient(p, **kw)
    b = TP.loss_gradient(p, checkpoints=True, **kw)
    np.testing.assert_array_equal(a.dL_dxv0, b.dL_dxv0)
    assert np.isfinite(a.dL_dB).all()
    # the failed allocation has left no error for the next call to report
    TP.solve(p, TP.Boris(), dt=kw["dt"], precision="fp32c", save_everystep=False)
    print("same")


# 3.1 GB of rows, which the context would keep, and 6.2 GB, which it would not
@pytest.mark.parametrize("n", [65536, 131072])
def test_without_room_for_the_trajectory(n):
    here = os.path.dirname(os.path.abspath(__file__))
    code = f"import sys; sys.path.insert(0, {here!r}); import conftest; import test_gpu_adjoint_memory as t; t.limited({n}, 1700)"
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=110,
                       env=dict(os.environ, GPU_SINGLE_ALLOC_PERCENT="1"))
    assert r.returncode == 0, r.stdout + r.stderr
    if "no limit" in r.stdout:
        pytest.skip("the runtime does not limit single allocations")
    assert "same" in r.stdout
