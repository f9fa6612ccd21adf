"""What the host code launches, over a HIP runtime on the host (fake_hip.c):
a launch that fails reaches the caller as an error, and the tuning overrides
set the launch shapes that they say."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

SETUP = """
import ctypes, sys
import numpy as np
from piny_amd import abi, water as w
from piny_amd.engine import Engine, PinyAmdError
fake = ctypes.CDLL(None)
"""
STEPS = SETUP + """
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
TILES = SETUP + """
c = w.small_config(w.SPC_FW, nmol=64, P=1, seed=1, kmax=14)  # a 32^3 grid
eng = Engine(c.system, c.x, c.y, c.z)
eng.set_positions(c.x, c.y, c.z)
eng.energy_control()
print(fake.fake_grid(b"k_pme_gather"))
"""
CELLS = SETUP + """
nmol, cell = int(sys.argv[1]), np.array(eval(sys.argv[2]))
L = w.density_box(nmol)
c = w.build_config(w.SPC_FW, nmol, L, 1, 1, w.Settings(kmax_ewd=10, kmax_pme=10))
eng = Engine(w.with_cell(c, cell / np.linalg.det(cell) ** (1 / 3) * L).system)
eng.set_positions(c.x, c.y, c.z)
eng.energy_control()
print(fake.fake_grid(b"k_cell_order") > 0)
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake_hip") / "fake_hip.so")
    subprocess.run(["gcc", "-O1", "-w", "-shared", "-fPIC", "-o", so, os.path.join(HERE, "fake_hip.c")], check=True)

    def run_(code, *args, **env):
        env = dict(os.environ, PYTHONPATH=ROOT, **env)
        env["LD_PRELOAD"] = " ".join(p for p in (so, os.environ.get("LD_PRELOAD")) if p)
        r = subprocess.run([sys.executable, "-c", code, *args], env=env, cwd=ROOT, capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0, r.stderr
        return r.stdout
    return run_


# the launches of two steps: chains, kick and drift before the forces, kick
# and chains after them; the last step's are the call's last launches
@pytest.mark.parametrize("kernel, nth", [("k_nhc_ckin", 1), ("k_nhc_ckin", 4), ("k_nhc_class", 1), ("k_nhc_class", 2),
                                         ("k_nhc_class", 4), ("k_nhc_kick", 1), ("k_nhc_kick", 2), ("k_nhc_kick", 4),
                                         ("k_mode_drift", 1), ("k_nhc_scale0", 2), ("k_pair", 2)])
def test_pimd_step_launch_fails(run, kernel, nth):
    assert run(STEPS, kernel, str(nth)).startswith("raised")


# one workgroup a tile: upper bounds left out are those of 16,16,8, all zero
# (or none given) is the choice by the kernels
@pytest.mark.parametrize("tile, ntile", [("16,16,8", 2 * 2 * 4), ("16", 2 * 2 * 4), ("8,8", 4 * 4 * 4),
                                         ("8,4,2", 4 * 8 * 16), ("0,16,8", 32 * 2 * 4), ("0,0,0", None), ("", None)])
def test_pme_tile_override(run, tile, ntile):
    if ntile is None:
        ntile = int(run(TILES))
        assert ntile != 2 * 2 * 4
    assert int(run(TILES, PMX_PME_TILE=tile)) == ntile


# the list is built by cells where they spare a site 6000 candidates, 2000 in
# a triclinic cell
HEXAGONAL = "((1.0, 0.5, 0.0), (0.0, 0.866, 0.0), (0.0, 0.0, 1.0))"


@pytest.mark.parametrize("nmol, cell, cells", [(2000, "np.eye(3)", False), (4000, "np.eye(3)", True),
                                               (1000, HEXAGONAL, False), (2000, HEXAGONAL, True),
                                               (2700, HEXAGONAL, True)])
def test_list_cells_rule(run, nmol, cell, cells):
    assert run(CELLS, str(nmol), cell).split() == [str(cells)]
