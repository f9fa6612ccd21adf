"""Force calls at the bead counts, grid sizes and box sizes where a kernel's
launch shape or branch changes, against the oracle."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from piny_amd import abi, water as w

pytestmark = pytest.mark.gpu

# FP64 results differ from the oracle by the order of sums only
FP64_TOL = 1e-9


def call(c, **kw):
    from piny_amd.engine import Engine
    flags = abi.PMX_EVAL_PIMD if c.system.pi_beads > 1 else 0
    eng = Engine(c.system, c.x, c.y, c.z, **kw)
    eng.set_positions(c.x, c.y, c.z)
    e, f = eng.energy_control(flags), eng.forces()
    eng.close()
    eo, fo, _ = Oracle(c.system, c.x, c.y, c.z).energy_control(c.x, c.y, c.z, flags)
    return e, f, eo, fo


def check(c, **kw):
    e, f, eo, fo = call(c, **kw)
    scale = max(abs(eo[k]) for k in abi.ENERGY_KEYS)
    assert e["nver"] == eo["nver"]
    for k in abi.ENERGY_KEYS:
        assert abs(e[k] - eo[k]) < FP64_TOL * scale, k
    assert np.abs(e["pvten"] - eo["pvten"]).max() < FP64_TOL * np.abs(eo["pvten"]).max()
    assert np.sqrt(((f - fo) ** 2).sum() / (fo ** 2).sum()) < FP64_TOL


# bead counts that divide a wavefront (lane exchanges) and that do not (LDS
# runs), up to one bead per lane and to more slots than rows
@pytest.mark.parametrize("P", [1, 2, 3, 6, 12, 40, 48, 64])
def test_partial_sums_per_bead_count(P):
    check(w.small_config(w.Q_TIP4P_F, nmol=30, P=P, seed=40 + P))
