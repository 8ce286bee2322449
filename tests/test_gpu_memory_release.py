"""Device memory that the library takes to be faster: cell copies that are not
wanted, copies and workspace given back on request and before an allocation
fails; the results stay the same bits."""
import os
import subprocess
import sys

import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd import _lib
from testparticle_amd.device import DeviceEnsemble

pytestmark = pytest.mark.gpu

L, M, N, NT = 1.0e8, 80, 9001, 300                # N * NT gathers build a copy: 98 MB, or two of them
COPY = M**3 * 192


def grid(seed, layout):
    A = np.random.default_rng(seed).normal(0.0, 1e-9, (3, M, M, M))
    A[2] += 5e-9
    return TP.GridField(A, *[np.arange(M) * (L / M)] * 3, bc=TP.PeriodicBC(), layout=layout)


def problem(kind, layout):
    B = grid(1, layout) if kind == "grid" else TP.LazyTimeInterpolator([0.0, 60.0], lambda i: grid(i, layout))
    rng = np.random.default_rng(5)
    xv = np.hstack([rng.uniform(0.0, L, (N, 3)), rng.normal(0.0, 1e6, (N, 3))])
    return TP.TraceProblem(xv, (0.0, NT * 0.3), (TP.qi / TP.mi, TP.mi, TP.ZeroField(), B, TP.ZeroField()))


def free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def run(p):
    """The bits of a solve and the device memory that it left taken."""
    e = DeviceEnsemble(p, TP.Boris(), p.u0, dt=0.3, save_everystep=False)
    before = free()
    e.run()
    return e.u.cpu().numpy().view(np.int64), before - free()


@pytest.mark.parametrize("kind", ["grid", "snapshots"])
def test_copies_that_are_not_wanted(kind):
    want, took = run(problem(kind, "nodes"))
    assert took > COPY // 2
    ctx = _lib.context(0)
    only, off = problem(kind, "nodes_only"), problem(kind, "nodes")
    h = off.p[3].handle(ctx)
    ctx.check(ctx.L.tpamd_field_grid_cells(ctx.h, h, 0))
    for p in (only, off):
        got, took = run(p)
        assert took < COPY // 2
        np.testing.assert_array_equal(got, want)
    if kind == "snapshots":
        with pytest.raises(_lib.ArgumentError):
            ctx.check(ctx.L.tpamd_field_grid_cells(ctx.h, h, 1))


@pytest.mark.parametrize("kind", ["grid", "snapshots"])
def test_trim_gives_back(kind):
    ctx = _lib.context(0)
    p = problem(kind, "nodes")
    TP.solve(p, TP.Boris(), dt=0.3, savestepinterval=10)               # staging buffer: 15 MB
    ctx.trim()
    want, took = run(p)                                                # the copy again
    assert took > COPY // 2
    before = free()
    ctx.trim()
    assert free() - before > COPY // 2
    for _ in range(2):
        np.testing.assert_array_equal(run(p)[0], want)
        np.testing.assert_array_equal(TP.solve(p, TP.Boris(), dt=0.3, save_everystep=False).u_all.reshape(want.shape)
                                      .view(np.int64), want)
    ctx.trim()
    ctx.trim()
    e = p.p[3](p.u0[:50, :3], t=20.0)
    run(p)
    np.testing.assert_array_equal(p.p[3](p.u0[:50, :3], t=20.0), e)
    p.p[3].release()                                                   # freed with its copy in place
    ctx.trim()


def limited():
    """In a process of its own whose single allocations are limited."""
    import torch
    try:
        torch.empty(4 << 30, dtype=torch.uint8, device="cuda")
        print("no limit")
        return
    except torch.OutOfMemoryError:
        pass
    p, other = problem("grid", "nodes"), problem("snapshots", "nodes")
    want, w2 = run(p)[0], run(other)[0]
    asked = problem("grid", "cells")
    w3 = run(asked)[0]
    before = free()
    with pytest.raises(_lib.DeviceError, match="out of memory"):
        TP.solve(TP.TraceProblem(p.u0[:1], p.tspan, p.p), TP.AdaptiveBoris(0.1), nout_cap=100_000_000)
    assert free() - before > 2 * COPY                                  # both fields' copies went before it failed
    for q, w in ((p, want), (other, w2), (asked, w3)):
        np.testing.assert_array_equal(run(q)[0], w)
    print("same")


def test_copies_go_before_an_allocation_fails():
    here = os.path.dirname(os.path.abspath(__file__))
    code = f"import sys; sys.path.insert(0, {here!r}); import conftest; import test_gpu_memory_release as t; t.limited()"
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=110,
                       env=dict(os.environ, GPU_SINGLE_ALLOC_PERCENT="1"))
    assert r.returncode == 0, r.stdout + r.stderr
    if "no limit" in r.stdout:
        pytest.skip("the runtime does not limit single allocations")
    assert "same" in r.stdout
