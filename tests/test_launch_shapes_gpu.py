"""Force calls at the bead counts, grid sizes and box sizes where a kernel's
launch shape or branch changes, against the oracle."""
import dataclasses

import numpy as np
import pytest

from oracle.oracle import Oracle
from piny_amd import abi, water as w

pytestmark = pytest.mark.gpu

# FP64 results differ from the oracle by the order of sums only
FP64_TOL = 1e-9


@pytest.fixture(scope="module", autouse=True)
def torch_first():
    """torch finds the GPU only if it looks before the library does."""
    import torch
    torch.cuda.init()


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


# tiles of the layout change: whole ones and a remainder, few and many beads
@pytest.mark.parametrize("nmol, P", [(2, 1), (64, 1), (65, 3), (4, 16), (7, 24), (33, 64)])
def test_positions_in_and_out(nmol, P):
    import torch
    from piny_amd.engine import Engine
    c = w.small_config(w.Q_TIP4P_F, nmol=nmol, P=P, seed=3)
    x = np.stack([v.reshape(P, -1) for v in (c.x, c.y, c.z)], 2)
    m = w.Q_TIP4P_F
    xg = x.reshape(P, nmol, 4, 3).copy()
    xg[:, :, 3] = sum(cf * xg[:, :, k] for k, cf in m.ghost[1])
    eng = Engine(c.system, c.x, c.y, c.z)
    eng.set_positions(c.x, c.y, c.z)
    host = eng.positions()
    eng.set_velocities(c.y, c.z, c.x)
    assert np.array_equal(eng.velocities(), x[:, :, [1, 2, 0]])
    dev = [torch.as_tensor(v, device="cuda") for v in (c.x, c.y, c.z)]
    torch.cuda.synchronize()
    eng.set_positions(c.x * 0.0, c.y, c.z)
    eng.set_positions_device(*[v.data_ptr() for v in dev])
    assert np.array_equal(eng.positions(), host)
    real = np.arange(4 * nmol) % 4 != 3
    assert np.array_equal(host[:, real], x[:, real])
    assert np.abs(host.reshape(P, nmol, 4, 3) - xg).max() < 1e-12
    eng.close()


# the FP64 table kernel: wavefronts sharing a site (few sites), a partial last
# workgroup, more sites than wavefronts, tables too short and too long for LDS
@pytest.mark.parametrize("nmol, P, nsplin", [(2, 1, 5000), (27, 1, 5000), (201, 2, 5000), (300, 2, 5000), (400, 4, 5000),
                                             (430, 1, 5000), (343, 1, 512), (700, 1, 511),
                                             (1400, 1, 5000), (64, 8, 7200), (64, 8, 6900)])
def test_pair_table_in_lds(nmol, P, nsplin):
    c = w.small_config(w.SPC_FW, nmol=nmol, P=P, seed=nmol)
    c.system.settings.nsplin = nsplin
    check(c)


# two sites at one place, in every bead: a pair inside the cutoff, evaluated
# past the start of its table, counted, and without a force of its own.  The
# cubic reaches back over 82 points (0.1 A at 0.0012 A), with weights of up to
# 82^3 / 2 = 3e5 on values rounded to 1e-16: 3e-11 of a table value.
@pytest.mark.parametrize("P", [1, 2])
@pytest.mark.parametrize("site", [0, 1])
def test_pair_at_no_distance(monkeypatch, P, site):
    from piny_amd.engine import Engine
    c = w.small_config(w.SPC_FW, nmol=64, P=P, seed=5)
    for v in (c.x, c.y, c.z):
        v = v.reshape(P, 64, 3)
        v[:, 7] += v[:, 3, site, None] - v[:, 7, site, None]
        v[:, 7, site] = v[:, 3, site]
    check(c)
    npair = []
    for mode in ("full", "half"):
        monkeypatch.setenv("PMX_PAIR_LIST", mode)
        eng = Engine(c.system, c.x, c.y, c.z)
        eng.set_positions(c.x, c.y, c.z)
        eng.energy_control()
        npair.append(eng.pair_count())
        eng.close()
    assert npair[0] == npair[1]


# Nose-Hoover chains: every length is a kernel of its own; the state against
# the oracle's integrator
@pytest.mark.parametrize("len_nhc", [1, 2, 3, 4, 5, 6, 7])
def test_chain_lengths(len_nhc):
    from piny_amd.engine import Engine
    c = w.small_config(w.Q_TIP4P_F, nmol=27, P=4, seed=9)
    par = abi.nhc_params(len_nhc=len_nhc)
    rng = np.random.default_rng(len_nhc)
    v = rng.normal(size=(3, c.x.size)) * 1e-4
    v.reshape(3, 4, -1)[:, :, c.system.ghost_atom] = 0.0
    eng = Engine(c.system, c.x, c.y, c.z)
    eng.set_positions(c.x, c.y, c.z)
    eng.set_velocities(*v)
    _, ec = eng.pimd_nvt(3, par)
    vel, x, chains = eng.velocities(), eng.positions(), eng.nhc_state()
    o = Oracle(c.system, c.x, c.y, c.z)
    v0 = v.reshape(3, 4, -1).transpose(1, 2, 0)
    xo, vo, st, _, eco = o.pimd_nvt(3, c.x, c.y, c.z, v0, params=par)
    assert np.abs(x - xo).max() < 1e-9 * np.abs(xo).max()
    assert np.abs(vel - vo).max() < 1e-9 * np.abs(vo).max()
    assert np.abs(chains - st).max() < 1e-9 * np.abs(st).max()
    assert abs(ec[3] - eco[3]) < 1e-9 * np.abs(eco).max()
    eng.close()


# the force list by cells and by the scan over every site, orthorhombic (FP32
# test first) and triclinic (none), rows that fill a queue and that do not
@pytest.mark.parametrize("mode", ["brute", "cells"])
@pytest.mark.parametrize("nmol, P, cell", [(2, 1, None), (65, 4, None), (300, 1, None), (700, 2, None),
                                           (300, 2, ((1.0, 0.15, 0.0), (0.0, 1.0, 0.1), (0.05, 0.0, 1.0)))])
def test_list_rows(monkeypatch, mode, nmol, P, cell):
    from piny_amd.engine import Engine
    monkeypatch.setenv("PMX_LIST", mode)
    rc = 3.0 if nmol > 2 else 2.0
    c = w.small_config(w.SPC_FW, nmol=nmol, P=P, seed=nmol, cutoff=rc)
    if cell is not None:
        c = w.with_cell(c, np.array(cell) * c.system.box)
    x, y, z = c.x + 40.0, c.y - 55.0, c.z * 1.0  # outside the cell
    flags = abi.PMX_EVAL_PIMD if P > 1 else 0
    eng = Engine(c.system, x, y, z)
    eng.set_positions(x, y, z)
    e = eng.energy_control(flags)
    o = Oracle(c.system, x, y, z)
    eo, fo, _ = o.energy_control(x, y, z, flags)
    assert e["nver"] == eo["nver"]
    f = eng.forces()
    assert np.sqrt(((f - fo) ** 2).sum() / (fo ** 2).sum()) < FP64_TOL
    for a, b in zip(eng.verlet_list(), o.verlet_list()):
        assert np.array_equal(a, b)
    eng.close()


# more sites in one cell than a workgroup orders, on a new context: the list
# comes from the build without cells; then a call on spread positions
@pytest.mark.parametrize("P", [1, 2])
def test_list_of_an_overfull_cell(monkeypatch, P):
    from piny_amd.engine import Engine
    monkeypatch.setenv("PMX_LIST", "cells")
    c = w.small_config(w.SPC_FW, nmol=700, P=P, seed=1, cutoff=3.0)
    crowd = np.tile(np.arange(2100) < 1200, P)
    x, y, z = (np.where(crowd, 2.0 + 0.02 * (v - v.mean()), v) for v in (c.x, c.y, c.z))
    flags = abi.PMX_EVAL_PIMD if P > 1 else 0
    eng = Engine(c.system, x, y, z)
    o = Oracle(c.system, x, y, z)
    for pos in ((x, y, z), (c.x, c.y, c.z)):
        eng.set_positions(*pos)
        e = eng.energy_control(flags)
        eo, fo, _ = o.energy_control(*pos, flags)
        assert e["nver"] == eo["nver"]
        for a, b in zip(eng.verlet_list(), o.verlet_list()):
            assert np.array_equal(a, b)
    f = eng.forces()
    assert np.sqrt(((f - fo) ** 2).sum() / (fo ** 2).sum()) < FP64_TOL
    eng.close()


# a crowd of sites of which not all interact (the oxygens of q-TIP4P/F have no
# charge): the reference's longest row is longer than the force list's
@pytest.mark.parametrize("mode", ["brute", "cells"])
def test_reference_list_of_a_crowd(monkeypatch, mode):
    from piny_amd.engine import Engine
    monkeypatch.setenv("PMX_LIST", mode)
    c = w.small_config(w.Q_TIP4P_F, nmol=230, seed=1, box=60.0, cutoff=5.0)
    x, y, z = (0.1 * (v - v.mean()) for v in (c.x, c.y, c.z))
    eng = Engine(c.system, x, y, z)
    eng.set_positions(x, y, z)
    e = eng.energy_control(0)
    o = Oracle(c.system, x, y, z)
    eo, _, _ = o.energy_control(x, y, z, 0)
    assert e["nver"] == eo["nver"]
    for a, b in zip(eng.verlet_list(), o.verlet_list()):
        assert np.array_equal(a, b)
    eng.close()


# PME: a bead's sort in one workgroup and in three launches, the matrix-core
# spread (10^5 items) and the LDS one, orders and grids with and without its
# tiles, FP64 and mixed (the mixed bars of the parity tests)
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("nmol, P, order, kmax", [(64, 1, 4, 6), (690, 1, 6, 10), (530, 64, 6, 10), (530, 64, 4, 14),
                                                  (530, 64, 8, 14), (600, 60, 7, 17), (90, 2, 9, 10),
                                                  (530, 64, 5, 8)])
def test_pme_bins_and_spread(prec, nmol, P, order, kmax):
    c = w.small_config(w.SPC_FW, nmol=nmol, P=P, seed=nmol + order, cutoff=2.5, kmax=kmax)
    c.system.settings.n_interp = order
    if prec == "fp64":
        return check(c)
    e, f, eo, fo = call(c, precision=abi.PMX_PREC_MIXED)
    scale = max(abs(eo[k]) for k in abi.ENERGY_KEYS)
    for k in abi.ENERGY_KEYS:
        assert abs(e[k] - eo[k]) < 1e-5 * scale, k
    assert np.sqrt(((f - fo) ** 2).sum() / (fo ** 2).sum()) < 1e-4


# every grid size with FFT kernels of its own, and one without (100), against
# the oracle's own transform of the same grid
@pytest.mark.parametrize("K", [12, 16, 20, 24, 32, 36, 40, 48, 60, 64, 72, 80, 96, 100])
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_fft_sizes(prec, K):
    if prec == "fp64" and K == 100:
        pytest.skip("a 100 x 100 FP64 plane and its twiddles exceed a workgroup's LDS")
    c = w.small_config(w.SPC_FW, nmol=64, P=2, seed=K, kmax=2 * (K // 4 - 1))
    c.system.settings.kmax_ewd = min(c.system.settings.kmax_ewd, K // 2 - 2)
    if prec == "fp64":
        check(c)
    else:
        e, f, eo, fo = call(c, precision=abi.PMX_PREC_MIXED)
        scale = max(abs(eo[k]) for k in abi.ENERGY_KEYS)
        assert abs(e["vrecip"] - eo["vrecip"]) < 1e-5 * scale
        assert np.sqrt(((f - fo) ** 2).sum() / (fo ** 2).sum()) < 1e-4


# the kernel between two force calls of the NVE integrator: one step (no half
# kick before), and several at once, one at a time and by the oracle's forces,
# with sites of a whole workgroup, of one more, and with ghosts
@pytest.mark.parametrize("model, nmol, nsteps", [(w.SPC_FW, 64, 1), (w.SPC_FW, 64, 2), (w.Q_TIP4P_F, 65, 5),
                                                 (w.SPC_FW, 86, 7)])
def test_nve_steps_at_once(model, nmol, nsteps):
    from piny_amd.engine import Engine
    from tests.test_md_nve import oracle_nve
    c = w.small_config(model, nmol=nmol, P=1, seed=nmol)
    out = []
    dt = 0.25 / abi.TIME_CONV
    for calls in ([nsteps], [1] * nsteps):
        eng = Engine(c.system, c.x, c.y, c.z)
        eng.set_positions(c.x, c.y, c.z)
        for n in calls:
            e, ke = eng.md_nve(n, dt)
        out.append((e, ke, eng.positions()[0], eng.velocities()[0], eng.forces()[0]))
        eng.close()
    e1, k1, x1, v1, f1 = oracle_nve(c, np.zeros((c.system.natm, 3)), nsteps, dt)
    scale = max(abs(e1[k]) for k in abi.ENERGY_KEYS)
    for e0, k0, x0, v0, f0 in out:
        for k in abi.ENERGY_KEYS:
            assert abs(e0[k] - e1[k]) < FP64_TOL * scale, k
        assert k1 > 0 and abs(k0 - k1) < FP64_TOL * k1
        for a, b in ((x0, x1), (v0, v1), (f0, f1)):
            assert np.sqrt(((a - b) ** 2).sum() / (b ** 2).sum()) < FP64_TOL


def equal_beads(one, P):
    """The one-bead configuration with P beads at its places."""
    return w.Config(dataclasses.replace(one.system, pi_beads=P), *(np.tile(v, P) for v in (one.x, one.y, one.z)))


def check_equal_beads(one, c, prec):
    """The call on P equal beads has the energies of one bead, and its forces
    / P on each."""
    from piny_amd.engine import Engine
    P = c.system.pi_beads
    eo, fo, _ = Oracle(one.system, one.x, one.y, one.z).energy_control(one.x, one.y, one.z, 0)
    eng = Engine(c.system, c.x, c.y, c.z, precision=abi.PMX_PREC_MIXED if prec == "mixed" else abi.PMX_PREC_FP64)
    eng.set_positions(c.x, c.y, c.z)
    e = eng.energy_control(abi.PMX_EVAL_PIMD if P > 1 else 0)
    f = eng.forces() * P
    eng.close()
    etol, ftol = (FP64_TOL, FP64_TOL) if prec == "fp64" else (1e-5, 1e-4)
    scale = max(abs(eo[k]) for k in abi.ENERGY_KEYS)
    assert e["nver"] == eo["nver"]
    for k in abi.ENERGY_KEYS:
        assert abs(e[k] - eo[k]) < etol * scale, k
    assert np.sqrt(((f - fo) ** 2).sum() / (P * (fo ** 2).sum())) < ftol


def rod_config(axis, nmol, P, edge=5.0, length=975.0):
    """Waters spread along a rod, its ends included: 1080 grid points along
    axis and 8 along the others; P beads all at the same places."""
    st = w.Settings(cutoff=2.4, skin=0.1, res_dist=2.0, rheal=0.5, alpha=3.5 / 2.4, kmax_ewd=8, kmax_pme=16)
    c = w.build_config(w.SPC_FW, nmol, w.density_box(nmol), 1, 11, st)
    e = np.full(3, edge)
    e[axis] = length
    to = np.random.default_rng(11).uniform(size=(nmol, 3)) * e
    to[:, axis] = (np.arange(nmol) + 0.5) * length / nmol
    x = np.stack([v.reshape(nmol, 3) for v in (c.x, c.y, c.z)], 2)
    x += to[:, None] / w.BOHR - x[:, :1]
    one = w.with_cell(w.Config(c.system, *(np.ascontiguousarray(x[..., d]).reshape(-1) for d in range(3))), np.diag(e))
    return one, equal_beads(one, P)


# grid axes past 1024 points, each axis in turn, the LDS and (10^5 items) the
# matrix-core spread, and a tile asked to be as long as the axis
@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("axis, nmol, P, tile", [(0, 60, 1, None), (1, 60, 1, None), (2, 60, 1, None), (0, 530, 64, None),
                                                 (1, 530, 64, None), (2, 530, 64, None), (2, 60, 1, "1,1,1080")])
def test_pme_long_axis(monkeypatch, prec, axis, nmol, P, tile):
    one, c = rod_config(axis, nmol, P)
    if tile:
        monkeypatch.setenv("PMX_PME_TILE", tile)
        one.system.settings.n_interp = 4
    assert sorted(Oracle(one.system, one.x, one.y, one.z).scalars()[10:13]) == [8, 8, 1080]
    check_equal_beads(one, c, prec)


# grids that are not cubes, under the matrix-core spread (10^5 items) and the
# LDS one: tiles wider along a than along b and the reverse, odd ones, and a
# triclinic cell
SHEAR = ((1.0, 0.15, 0.0), (0.0, 1.0, 0.1), (0.05, 0.0, 1.0))


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("P", [64, 2])
@pytest.mark.parametrize("grid, order, shear", [((48, 48, 64), 6, None), ((48, 40, 64), 6, None), ((36, 48, 40), 6, None),
                                                ((40, 36, 48), 8, None), ((48, 40, 36), 4, None), ((36, 40, 64), 6, SHEAR)])
def test_pme_grids_not_cubic(prec, P, grid, order, shear):
    nmol = 530
    k = np.array(grid) / 4 - 1
    kpme = round(2 * k.prod() ** (1 / 3))
    st = w.Settings(cutoff=2.5, skin=0.5, alpha=1.0, kmax_ewd=8, kmax_pme=kpme, n_interp=order)
    L = w.density_box(nmol)
    c = w.build_config(w.SPC_FW, nmol, L, 1, 21, st)
    cell = np.diag(L * k / k.prod() ** (1 / 3)) @ np.array(shear or np.eye(3))
    # molecules at the fractions of the cell that they have of the cube
    x = np.stack([v.reshape(nmol, 3) for v in (c.x, c.y, c.z)], 2)
    x += (x[:, :1] * w.BOHR / L) @ cell.T / w.BOHR - x[:, :1]
    one = w.with_cell(w.Config(c.system, *(np.ascontiguousarray(x[..., d]).reshape(-1) for d in range(3))), cell)
    assert tuple(Oracle(one.system, one.x, one.y, one.z).scalars()[10:13]) == grid
    check_equal_beads(one, equal_beads(one, P), prec)
