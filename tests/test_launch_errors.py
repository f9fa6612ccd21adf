"""A kernel launch that fails in a call reaches the caller as an error: the
host code over a HIP runtime on the host (fake_hip.c) that fails the n-th
launch of a kernel."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

CALLS = """
import ctypes, sys
import numpy as np
from piny_amd import abi, water as w
from piny_amd.engine import Engine, PinyAmdError

fake = ctypes.CDLL(None)
kernel, nth = sys.argv[1].encode(), int(sys.argv[2])
c = w.small_config(w.Q_TIP4P_F, nmol=8, P=4, seed=1, cutoff=2.0)
eng = Engine(c.system, c.x, c.y, c.z)
eng.set_positions(c.x, c.y, c.z)
par = abi.nhc_params(len_nhc=3)
eng.pimd_nvt(2, par)  # no failure
fake.fake_fail(kernel, nth)
try:
    eng.pimd_nvt(2, par)
    print("returned")
except PinyAmdError as e:
    print("raised", e)
"""


@pytest.fixture(scope="module")
def preload(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake_hip") / "fake_hip.so")
    subprocess.run(["gcc", "-O1", "-w", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.c")], check=True)
    return so


# the launches of two steps: chains, kick and drift before the forces, kick
# and chains after them; the last step's are the call's last launches
@pytest.mark.parametrize("kernel, nth", [("k_nhc_ckin", 1), ("k_nhc_ckin", 4), ("k_nhc_class", 1), ("k_nhc_class", 2),
                                         ("k_nhc_class", 4), ("k_nhc_kick", 1), ("k_nhc_kick", 2), ("k_nhc_kick", 4),
                                         ("k_mode_drift", 1), ("k_nhc_scale0", 2), ("k_pair", 2)])
def test_pimd_step_launch_fails(preload, kernel, nth):
    env = dict(os.environ, PYTHONPATH=ROOT)
    env["LD_PRELOAD"] = " ".join(p for p in (preload, os.environ.get("LD_PRELOAD")) if p)
    r = subprocess.run([sys.executable, "-c", CALLS, kernel, str(nth)], env=env, cwd=ROOT, capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    assert r.stdout.startswith("raised"), r.stdout
