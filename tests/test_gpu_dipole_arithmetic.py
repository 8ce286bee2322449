"""The dipole kernel's own division and square root, and particles whose field
has components that are exactly zero at every step."""
import json
import os
import subprocess

import pytest

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
