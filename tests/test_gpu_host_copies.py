"""Host-array solves against device-array solves at the sizes where the copies
change: one piece, the limit of the staged copy to the device, pieces that end
inside an array, more pieces than the pinned memory holds at once."""
import numpy as np
import pytest

import testparticle_amd as TP
from testparticle_amd.device import DeviceEnsemble

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own_steps", [False, True])
@pytest.mark.parametrize("n,saves", [(1, 0), (1, 1), (3, 4680), (4095, 1), (9361, 1), (9363, 1), (10917, 1), (10923, 1),
                                     (20011, 3), (30011, 9)])
def test_host_and_device_arrays_agree(n, saves, own_steps):
    rng = np.random.default_rng(n)
    xv = rng.normal(0.0, 1.0, (n, 6)) * [1, 1, 1, 1e5, 1e5, 1e5]
    nt = max(saves, 2)
    prob = TP.TraceProblem(xv, (0.0, nt * 0.1), (TP.qi / TP.mi, TP.mi, TP.UniformField([1e-4, 0.0, -2e-4]),
                                                 TP.UniformField([2e-9, 0.0, 1e-8]), TP.ZeroField()))
    kw = dict(dt=0.1, save_everystep=saves > 1, save_start=saves > 0, save_end=False, savestepinterval=1)
    if own_steps:
        kw.update(dts=rng.uniform(0.05, 0.1, n), nsteps=nt, dt=None)
    for _ in range(2):                                    # the second call meets used pieces
        a = TP.solve(prob, TP.Boris(), **kw)
    d = DeviceEnsemble(prob, TP.Boris(), xv, **kw)
    st = d.run()
    lengths = d.len.cpu().numpy()
    np.testing.assert_array_equal(a.lengths, lengths)
    np.testing.assert_array_equal(a.retcodes, d.ret.cpu().numpy())
    assert a.stats.particle_steps == st.particle_steps == n * nt
    k = int(lengths.max())
    assert (lengths == k).all() and k == a.u_all.shape[1]
    if k:
        np.testing.assert_array_equal(a.u_all.view(np.int64), d.u.cpu().numpy()[:, :k].view(np.int64))
        np.testing.assert_array_equal(a.t_all.view(np.int64), d.t.cpu().numpy()[:, :k].view(np.int64))
