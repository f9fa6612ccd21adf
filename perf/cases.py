"""What this framework is timed on: the force calls and integrator runs that a
user's program makes, through piny_amd's public entry points.

A case is a dict of plain values.  ``kind`` says which program it is:

* ``force``  a program that holds the bead positions on the GPU (its own
  integrator, a sampler, a learned potential's trainer): positions in
  (``set_positions_device``), one force call, energies and the device forces
  out.  ``modes`` adds the normal-mode forces and springs that a PIMD
  integrator asks for; ``rebuild`` makes a new Verlet list, as every call on
  an unrelated configuration does; ``respa`` is the short-range call of a
  multiple-time-step integrator.
* ``batch``  many uneven boxes in one call.
* ``nve``, ``pimd``  the device integrators run for some steps from given
  positions and velocities, the state read back.
* ``grad``   the force call as a torch function, forward and backward, with the
  gradients of the positions and of the water model's parameters.

``box`` settings follow the repository's uneven-box workload (0.997 g/cm^3,
r_c = min(9 A, L/2 - 0.05 A), alpha = 3.5 / r_c, a PME grid of about 1 A),
which also gives the 64^3 grid of the 4096-molecule box.
"""
import dataclasses
import math

import numpy as np
import torch

from piny_amd import abi, autograd, water
from piny_amd.engine import Batch, Engine

MODELS = {"spc_fw": water.SPC_FW, "q_tip4p_f": water.Q_TIP4P_F}
PRECISION = {"fp64": (abi.PMX_PREC_FP64, abi.PMX_PAIR_TABLE), "direct": (abi.PMX_PREC_FP64, abi.PMX_PAIR_DIRECT),
             "mixed": (abi.PMX_PREC_MIXED, abi.PMX_PAIR_TABLE)}
# the short-range call: step counts of the reference's q-TIP4P/F example
RESPA = {"respa_lrf": 4, "respa_torsion": 1, "respa_intra": 2, "respa_pimd": 5}
E_KEYS = ("vintert", "vintrat", "vreal", "vvdw", "vcoul", "vlong", "vrecip", "vself", "vbgr", "vecor", "vbond",
          "vbend", "kin_harm", "pi_ke_prim", "pi_ke_vir")


def listed():
    f = {"kind": "force", "modes": False, "rebuild": False, "respa": False}
    return [
        # the smallest box a user runs (64 molecules, classical): launches and waits are the call
        dict(f, name="spc64_p1_fp64", model="spc_fw", nmol=64, beads=1, prec="fp64"),
        # classical MD of the usual small box on the device integrator
        dict(name="nve_spc256", kind="nve", model="spc_fw", nmol=256, beads=1, prec="fp64", steps=20),
        # one large classical box, an odd molecule count: a single bead has to fill the GPU
        dict(f, name="spc5003_p1_fp64", model="spc_fw", nmol=5003, beads=1, prec="fp64"),
        # scoring unrelated path-integral configurations: every call builds its list
        dict(f, name="tip1024_p8_rebuild_fp64", model="q_tip4p_f", nmol=1024, beads=8, prec="fp64", rebuild=True),
        # PIMD NVT on the device integrator, chains included
        dict(name="pimd_spc343_p16", kind="pimd", model="spc_fw", nmol=343, beads=16, prec="fp64", steps=5),
        # the benchmark box: a PIMD step's force call in mixed precision ...
        dict(f, name="tip4096_p32_mixed", model="q_tip4p_f", nmol=4096, beads=32, prec="mixed", modes=True),
        # ... and in the reference's arithmetic
        dict(f, name="tip4096_p32_fp64", model="q_tip4p_f", nmol=4096, beads=32, prec="fp64", modes=True),
        # a ragged one: odd molecule count, a bead count that is no power of two
        dict(f, name="tip733_p6_mixed", model="q_tip4p_f", nmol=733, beads=6, prec="mixed", modes=True),
        # the largest: 36003 sites, 16 beads, a grid of 72 points a side
        dict(f, name="spc12001_p16_mixed", model="spc_fw", nmol=12001, beads=16, prec="mixed"),
        # the short-range call between two full ones of a multiple-time-step run
        dict(f, name="respa_tip1500_p16_mixed", model="q_tip4p_f", nmol=1500, beads=16, prec="mixed", modes=True,
             respa=True),
        # uneven boxes in one call (replicas, umbrella windows)
        dict(name="batch_spc_x12_mixed", kind="batch", model="spc_fw", nmol=1536, beads=32, boxes=12, prec="mixed"),
        # fitting the water model: energies, forces and parameter gradients
        dict(name="grad_tip512_p8_fp64", kind="grad", model="q_tip4p_f", nmol=512, beads=8, prec="fp64"),
    ]


def draw(rng):
    kind = rng.choice(["force"] * 6 + ["nve", "pimd", "batch", "grad"])
    model = rng.choice(["spc_fw", "q_tip4p_f"])
    prec = rng.choice(["fp64", "mixed"])

    def size(lo, hi):
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))

    beads = rng.choice([1, 1, 2, 4, 6, 8, 12, 16, 24, 32, 64])
    cap = 16384 // beads if prec == "fp64" else 49152 // beads  # molecules x beads, below the largest case's cost
    if kind == "nve":
        return dict(kind=kind, model=model, nmol=size(64, 1500), beads=1, prec="fp64", steps=rng.randint(5, 20))
    if kind == "pimd":
        beads = rng.choice([4, 8, 16, 32])
        return dict(kind=kind, model=model, nmol=size(64, 8192 // beads), beads=beads, prec="fp64",
                    steps=rng.randint(2, 6))
    if kind == "batch":
        return dict(kind=kind, model="spc_fw", nmol=size(200, 1536), beads=rng.choice([8, 16, 32]),
                    boxes=rng.randint(3, 12), prec=prec)
    if kind == "grad":
        beads = rng.choice([1, 4, 8])
        return dict(kind=kind, model=model, nmol=size(64, 700), beads=beads, prec="fp64")
    respa = beads > 1 and rng.random() < 0.2
    return dict(kind=kind, model=model, nmol=size(150 if respa else 64, min(9000, max(200, cap))), beads=beads,
                prec="direct" if prec == "fp64" and rng.random() < 0.2 else prec,
                modes=beads > 1 and rng.random() < 0.6, rebuild=rng.random() < 0.2, respa=respa)


def _settings(nmol, respa=False):
    """r_c, alpha and the PME grid of a box of nmol molecules (see above)."""
    L = water.density_box(nmol)
    rc = min(9.0, 0.5 * L - 0.05)
    K = min(water.RADIX_SIZES, key=lambda r: abs(r - L))
    kp = max(2, 2 * (K // 4 - 1))
    extra = dict(RESPA, res_dist=min(5.0, rc - 1.0)) if respa else {}
    return L, water.Settings(cutoff=rc, alpha=3.5 / rc, kmax_ewd=min(kp, K // 2 - 2), kmax_pme=kp, **extra)


def _config(case, seed):
    L, st = _settings(case["nmol"], case.get("respa", False))
    cfg = water.build_config(MODELS[case["model"]], case["nmol"], L, case["beads"], seed, st)
    if case["beads"] > 1:
        return cfg
    # a classical box's molecules come out of the builder at their equilibrium
    # geometry: thermal displacements of the real sites, as in any running system
    m, rng = cfg.system.model, np.random.Generator(np.random.PCG64(seed + 55))
    x = np.stack([cfg.x, cfg.y, cfg.z], 1).reshape(case["nmol"], len(m.sites), 3)
    x = x + rng.normal(size=x.shape) * 0.03 / water.BOHR
    if m.ghost is not None:
        x[:, m.ghost[0]] = sum(c * x[:, k] for k, c in m.ghost[1])
    return water.Config(cfg.system, *(np.ascontiguousarray(x[:, :, d].reshape(-1)) for d in range(3)))


def _batch_configs(case, seed):
    """Molecule counts spread over a factor of 24 up to nmol, bead counts up
    to beads, as in the uneven-box workload."""
    rng = np.random.Generator(np.random.PCG64(100 + case["boxes"]))  # the boxes' sizes belong to the case
    lo = max(64, case["nmol"] // 24)
    n = np.exp(rng.uniform(math.log(lo), math.log(case["nmol"]), case["boxes"])).astype(int)
    P = rng.choice(np.array([p for p in (1, 4, 8, 16, 32) if p <= case["beads"]]), case["boxes"])
    return [_config(dict(case, nmol=int(n[k]), beads=int(P[k])), seed + 1000 * k) for k in range(case["boxes"])]


def _velocities(system, P, seed):
    """Maxwell velocities of the modes (masses as the integrators use them)."""
    rng = np.random.Generator(np.random.PCG64(seed + 77))
    m = np.asarray(system.mass)[None, :] * _mode_mass(P)[:, None]
    v = rng.normal(size=(3, P, system.natm)) * np.sqrt(system.settings.temperature / water.BOLTZ / m)
    v[:, :, system.ghost_atom] = 0.0
    return [np.ascontiguousarray(c.reshape(-1)) for c in v]


def _mode_mass(P):
    if P == 1:
        return np.ones(1)
    f = np.zeros(P)
    for k in range(1, P // 2):
        f[2 * k - 1] = f[2 * k] = (1.0 - math.cos(2.0 * math.pi * k / P)) * 4.0 * P
    f[P - 1] = 4.0 * P
    f[0] = 1.0
    return f


class _DeviceArray:
    """A device array of an engine as torch sees it; a tensor made of it holds
    on to the engine, whose memory it is."""

    def __init__(self, eng, ptr, n):
        self.engine = eng
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (ptr, False), "version": 2}


def _engine(case, cfg):
    prec, pair = PRECISION[case["prec"]]
    eng = Engine(cfg.system, cfg.x, cfg.y, cfg.z, precision=prec, pair_eval=pair)
    if case.get("respa"):
        eng.set_respa(abi.respa_params(cfg.system))
    pos = [torch.as_tensor(v, device="cuda") for v in (cfg.x, cfg.y, cfg.z)]
    n = cfg.system.natm * cfg.system.pi_beads
    frc = [torch.as_tensor(_DeviceArray(eng, p, n), device="cuda") for p in eng.forces_device()]
    return eng, pos, frc


def _flags(case, P):
    fl = abi.PMX_EVAL_PIMD if P > 1 else 0
    fl |= abi.PMX_EVAL_MODE_FORCES if case["modes"] else 0
    fl |= abi.PMX_EVAL_FORCE_LIST if case["rebuild"] else 0
    fl |= abi.PMX_EVAL_RES_INTER | abi.PMX_EVAL_NO_FULL_INTER if case["respa"] else 0
    return fl


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        cfgs = _batch_configs(case, seed)
        parts = [_engine(case, c) for c in cfgs]
        for eng, pos, _ in parts:
            torch.cuda.synchronize()
            eng.set_positions_device(*[p.data_ptr() for p in pos])
        return {"kind": kind, "parts": parts, "batch": Batch([p[0] for p in parts])}
    cfg = _config(case, seed)
    if kind == "force":
        eng, pos, frc = _engine(case, cfg)
        torch.cuda.synchronize()
        return {"kind": kind, "eng": eng, "pos": pos, "frc": frc, "flags": _flags(case, case["beads"])}
    prec, pair = PRECISION[case["prec"]]
    eng = Engine(cfg.system, cfg.x, cfg.y, cfg.z, precision=prec, pair_eval=pair)
    st = {"kind": kind, "eng": eng, "pos": (cfg.x, cfg.y, cfg.z)}
    if kind in ("nve", "pimd"):
        st["vel"] = _velocities(cfg.system, case["beads"], seed)
        st["steps"] = case["steps"]
    if kind == "pimd":
        st["nhc"] = abi.nhc_params(gamma_adb=1.0)
        st["chains"] = np.zeros(abi.nhc_state_size(eng.N, eng.P, st["nhc"].len_nhc))
    if kind == "grad":
        p = np.stack([v.reshape(eng.P, eng.N) for v in (cfg.x, cfg.y, cfg.z)], 2)
        st["x"] = torch.as_tensor(p, device="cuda").requires_grad_(True)
        st["params"] = {k: v.requires_grad_(True) for k, v in autograd.water_params(cfg.system.model).items()}
        torch.cuda.synchronize()
    return st


def _energies(e):
    return {"energies": np.array([e[k] for k in E_KEYS]), "pvten": e["pvten"], "pvten_tot": e["pvten_tot"],
            "nver": e["nver"]}


def _stacked(out, forces):
    return {**{k: None if out[0][k] is None else np.stack([o[k] for o in out]) for k in out[0]}, "forces": forces}


def run(state):
    kind, eng = state["kind"], state.get("eng")
    if kind == "force":
        eng.set_positions_device(*[p.data_ptr() for p in state["pos"]])
        return {**_energies(eng.energy_control(state["flags"])), "forces": state["frc"]}
    if kind == "batch":
        for e, pos, _ in state["parts"]:
            e.set_positions_device(*[p.data_ptr() for p in pos])
        out = state["batch"].energy_control()
        return _stacked([_energies(o) for o in out], [p[2] for p in state["parts"]])
    if kind == "nve":
        eng.set_positions(*state["pos"])
        eng.set_velocities(*state["vel"])
        eng.energy_control()
        e, ke = eng.md_nve(state["steps"], 0.5 / abi.TIME_CONV)
        return {**_energies(e), "kinetic": ke, "x": eng.positions(), "v": eng.velocities(), "f": eng.forces()}
    if kind == "pimd":
        eng.set_positions(*state["pos"])
        eng.set_velocities(*state["vel"])
        eng.set_nhc_state(state["chains"], state["nhc"].len_nhc)
        e, econs = eng.pimd_nvt(state["steps"], state["nhc"])
        return {**_energies(e), "econs": econs, "x": eng.positions(), "v": eng.velocities(), "f": eng.forces(),
                "chains": eng.nhc_state()}
    x, params = state["x"], state["params"]
    x.grad = None
    for p in params.values():
        p.grad = None
    e = autograd.water_energy(eng, x, params)
    e.sum().backward()
    return {"energy": e.detach(), "x": x.grad, **{k: p.grad for k, p in params.items()}}


# --- what a pass cannot do without ---------------------------------------------

def _grid(nmol):
    L = water.density_box(nmol)
    return min(water.RADIX_SIZES, key=lambda r: abs(r - L))


def _box_work(model, nmol, P, respa=False):
    """Bytes: positions in, forces out.  Flops: every site pair inside the
    cutoff once per bead (45 for separation, r, erfc term, force and sums),
    and order-6 PME: weights, spread and gather (8 n^3 + 150 per charge) and
    two real transforms of the grid."""
    sites, terms, charges = (3, 9, 3) if model == "spc_fw" else (4, 10, 3)
    L, st = _settings(nmol, respa)
    rc = st.res_dist if respa else st.cutoff
    mol_pairs = nmol * (nmol / L ** 3) * (4.0 / 3.0) * math.pi * rc ** 3 / 2
    flops = mol_pairs * terms * 45.0
    if not respa:
        K = _grid(nmol)
        flops += charges * nmol * (8 * 216 + 150) + 2 * 2.5 * K ** 3 * math.log2(K ** 3)
    return {"bytes": 48.0 * sites * nmol * P, "flops": flops * P}


def work(case):
    if case["kind"] == "batch":
        parts = [(c.system.nmol, c.system.pi_beads) for c in _batch_sizes(case)]
        w = [_box_work(case["model"], n, P) for n, P in parts]
        return {k: sum(v[k] for v in w) for k in ("bytes", "flops")}
    w = _box_work(case["model"], case["nmol"], case["beads"], case.get("respa", False))
    calls = case.get("steps", 0) + 1
    return {k: v * calls for k, v in w.items()}


def _batch_sizes(case):
    rng = np.random.Generator(np.random.PCG64(100 + case["boxes"]))
    lo = max(64, case["nmol"] // 24)
    n = np.exp(rng.uniform(math.log(lo), math.log(case["nmol"]), case["boxes"])).astype(int)
    P = rng.choice(np.array([p for p in (1, 4, 8, 16, 32) if p <= case["beads"]]), case["boxes"])

    @dataclasses.dataclass
    class _S:
        nmol: int
        pi_beads: int

    @dataclasses.dataclass
    class _C:
        system: _S
    return [_C(_S(int(a), int(b))) for a, b in zip(n, P)]


# --- the same numbers in 64 bits, written out in torch ---------------------------

# PINY's erfc polynomial in t = 1 / (1 + p a r), times exp(-(a r)^2)
ERF_P = 0.3614
ERF_E = (0.2041422096422003, 0.1997535956961481, 0.2213176596405576, 0.03360430734640255, 0.4732592578721755,
         -0.509078520069735, 0.6772631491947646, -0.369912979092217, 0.06965131976970335)


def _erfc(u):
    """(erfc, d erfc/du) of the polynomial."""
    t = 1.0 / (1.0 + ERF_P * u)
    g, dg = torch.zeros_like(u), torch.zeros_like(u)
    for k in range(9, 0, -1):
        dg = dg * t + g
        g = g * t + ERF_E[k - 1]
    dg = dg * t + g          # d/dt of t * g(t)
    g = g * t
    ex = torch.exp(-u * u)
    return g * ex, -dg * ex * ERF_P * t * t - 2.0 * u * g * ex


def _switch(r, rc, heal):
    b = ((r - rc + heal) / heal).clamp(0.0, 1.0)
    return 1.0 + b * b * (2.0 * b - 3.0), 6.0 * b * (b - 1.0) / heal


class _Exact:
    """Energies, virials and forces of one box, all beads, in FP64."""

    def __init__(self, cfg, respa=False, modes=False, sums=True):
        s, self.dev = cfg.system, "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=self.dev)
        self.s, self.P, self.N, self.modes, self.respa = s, s.pi_beads, s.natm, modes, respa
        st = s.settings
        self.ns = len(s.model.sites)
        self.L, self.V = s.hmat[0], s.hmat[0] * (s.hmat[0] * s.hmat[0])
        self.al = s.ewald_alpha / self.V ** (1.0 / 3.0)
        self.rc, self.heal = st.cutoff / water.BOHR, st.rheal / water.BOHR
        self.rr = st.res_dist / water.BOHR
        self.q, self.mass = t(s.q), t(s.mass)
        oxy = int(np.argmax(s.inter_label == 2))
        self.eps, self.sig = float(s.inter_eps[oxy]), float(s.inter_sig[oxy])
        self.T = st.temperature
        self.nreal = self.N - len(s.ghost_atom)
        nsteps = (st.respa_pimd or 1), (st.respa_intra or 1) * (st.respa_torsion or 1), (st.respa_lrf or 1)
        self.w_tra, self.w_res = (float(nsteps[0]), float(nsteps[0] * nsteps[1])) if respa else (1.0, 1.0)
        self.w_ter = self.w_res * nsteps[2]
        self.kspace()
        self.sums = {}

    # -- PME tables
    def kspace(self):
        st, L, V = self.s.settings, self.L, self.V
        K = _grid(self.s.nmol)
        self.K, kmax = K, st.kmax_ewd
        hi, tpi = (L * L) / V, 2.0 * math.pi
        rv = V ** (-2.0 / 3.0)
        ecut = math.pi * .5 * math.pi * float(kmax * kmax) * rv
        kv = int(2.0 * (math.sqrt(ecut * .5) / (math.pi * hi)))
        n = np.fft.fftfreq(K, 1.0 / K)
        g = (n * hi) * tpi
        m = np.arange(K)
        b = sum(c * np.exp(2j * math.pi * m * k / K)
                for k, c in enumerate(np.array([1.0, 26.0, 66.0, 26.0, 1.0]) / 120.0))
        bw = 1.0 / np.abs(b) ** 2
        Ha = K // 2 + 1
        gz, gy, gx = np.meshgrid(g, g, np.abs(g[:Ha]), indexing="ij")
        nz, ny, nx = np.meshgrid(n, n, np.abs(n[:Ha]), indexing="ij")
        g2 = gx * gx + gy * gy + gz * gz
        ok = (g2 * .5 <= ecut * 4.0) & (np.maximum(np.maximum(np.abs(nx), np.abs(ny)), np.abs(nz)) <= kv) & (g2 > 0)
        W = np.where(ok, np.exp(-g2 / (4 * self.al ** 2)) / (np.where(ok, g2, 1.0) * (V / (4 * math.pi))), 0.0)
        W = W * bw[:, None, None] * bw[None, :, None] * bw[None, None, :Ha]
        half = np.where(np.arange(Ha) == 0, 0.5, 1.0)[None, None, :]
        f = lambda a: torch.as_tensor(a, device=self.dev)
        self.W, self.Wh, self.gv, self.g2 = f(W), f(W * half), [f(gx), f(gy), f(gz)], f(np.where(g2 > 0, g2, 1.0))
        self.kcut = math.sqrt(2.0 * (4.0 * ecut))
        u = torch.tensor(self.kcut / (2.0 * self.al), dtype=torch.float64)
        self.self_erf = 1.0 - float(_erfc(u)[0])

    # -- one configuration [P, N, 3] with the image reference xm [N, 3]
    def pairs(self, x, xm):
        L, rcut = self.L, (self.rr if self.respa else self.rc)
        ref = xm if self.P > 1 else x[0]
        u = (x - ref).norm(dim=2).max()
        lim = rcut + 2.0 * float(u) + 1e-6
        mol = torch.arange(self.N, device=self.dev) // self.ns
        oxy = torch.as_tensor(np.asarray(self.s.atm_type) == 0, device=self.dev)
        chg = self.q != 0
        ii, jj = [], []
        for lo in range(0, self.N, 1024):
            a = torch.arange(lo, min(lo + 1024, self.N), device=self.dev)
            d = ref[a][:, None, :] - ref[None, :, :]
            d -= L * torch.round(d / L)
            hit = (d.square().sum(2) < lim * lim) & (mol[a][:, None] < mol[None, :])
            hit &= (chg[a][:, None] & chg[None, :]) | (oxy[a][:, None] & oxy[None, :])
            k = hit.nonzero()
            ii.append(k[:, 0] + lo)
            jj.append(k[:, 1])
        i, j = torch.cat(ii), torch.cat(jj)
        P, rep = self.P, {"vvdw": 0.0, "vcoul": 0.0, "a12": 0.0, "a6": 0.0}
        f, vir = torch.zeros_like(x), torch.zeros(3, 3, dtype=x.dtype, device=self.dev)
        eb = {k: torch.zeros(P, dtype=x.dtype, device=self.dev) for k in rep}
        step = max(1, 6_000_000 // P)
        for lo in range(0, len(i), step):
            a, b = i[lo:lo + step], j[lo:lo + step]
            d0 = ref[a] - ref[b]
            sh = L * torch.round(d0 / L)
            d = x[:, a] - x[:, b] - sh
            r2 = d.square().sum(2)
            r = r2.sqrt()
            inside = r < rcut
            rs = torch.where(inside, r, torch.full_like(r, rcut))
            sw, dsw = _switch(rs, self.rc, self.heal)
            qq = (self.q[a] * self.q[b])
            er, der = _erfc(self.al * rs)
            vc, dvc = er / rs, self.al * der / rs - er / (rs * rs)
            lj = (oxy[a] & oxy[b]).to(x.dtype)
            s6 = (self.sig / rs) ** 6
            vl = 4.0 * self.eps * s6 * (s6 - 1.0)
            dvl = -24.0 * self.eps * s6 * (2.0 * s6 - 1.0) / rs
            m = inside.to(x.dtype)
            dv = (qq * (dvc * sw + vc * dsw) + lj * (dvl * sw + vl * dsw)) * m
            eb["vcoul"] += (qq * vc * sw * m).sum(1)
            eb["vvdw"] += (lj * vl * sw * m).sum(1)
            eb["a12"] += (lj * 4.0 * self.eps * s6 * s6 * sw * m).sum(1)
            eb["a6"] += (lj * 4.0 * self.eps * s6 * sw * m).sum(1)
            if self.respa:
                dv = dv * _switch(rs, self.rr, self.heal)[0] * self.w_res
            fv = d * (-dv / rs)[:, :, None]
            f.index_add_(1, a, fv)
            f.index_add_(1, b, -fv)
            vir += torch.einsum("pna,pnb->ab", d, fv)
        return eb, f, vir

    def recip(self, x):
        K, P = self.K, self.P
        c = (self.q != 0).nonzero()[:, 0]
        q = self.q[c]
        f = torch.zeros_like(x)
        vir = torch.zeros(3, 3, dtype=x.dtype, device=self.dev)
        e = torch.zeros(P, dtype=x.dtype, device=self.dev)
        m = torch.arange(6, device=self.dev)
        for b in range(P):
            s = x[b, c] / self.L
            s = (s - torch.floor(s)) * K
            ig = torch.floor(s)
            fr = s - ig
            w, dw = self.spline(fr)                       # [n, 3, 6], support ig - 5 + m
            idx = (ig[:, :, None].long() - 5 + m) % K
            wx, wy, wz = w[:, 0], w[:, 1], w[:, 2]
            flat = ((idx[:, 2, :, None, None] * K + idx[:, 1, None, :, None]) * K + idx[:, 0, None, None, :])
            val = (q[:, None] * wz)[:, :, None, None] * wy[:, None, :, None] * wx[:, None, None, :]
            grid = torch.zeros(K ** 3, dtype=x.dtype, device=self.dev)
            grid.index_add_(0, flat.reshape(-1), val.reshape(-1))
            S = torch.fft.rfftn(grid.view(K, K, K))
            s2 = self.Wh * (S.real ** 2 + S.imag ** 2)
            e[b] = s2.sum()
            pre = -2.0 * s2 * (self.g2 / (4 * self.al ** 2) + 1.0) / self.g2
            for a1 in range(3):
                for a2 in range(3):
                    # the half a' = 0 plane holds both signs of (b, c)
                    vir[a1, a2] += (pre * self.gv[a1] * self.gv[a2]).sum()
                vir[a1, a1] += e[b]
            phi = torch.fft.irfftn(self.W * S, s=(K, K, K)).reshape(-1) * float(K) ** 3
            ph = phi[flat]
            g = torch.stack([torch.einsum("nzyx,nz,ny,nx->n", ph, wz, wy, dw[:, 0]),
                             torch.einsum("nzyx,nz,ny,nx->n", ph, wz, dw[:, 1], wx),
                             torch.einsum("nzyx,nz,ny,nx->n", ph, dw[:, 2], wy, wx)], 1)
            f[b, c] = -(q * K / self.L)[:, None] * g
        return e, f, vir

    @staticmethod
    def spline(fr):
        """Order-6 cardinal B-spline weights of the points ig - 5 + m, and
        their derivatives (the differences of order 5)."""
        w = [fr, 1.0 - fr]                                # order 2: M2(fr), M2(fr + 1)
        for o in range(3, 7):
            if o == 6:
                z = torch.zeros_like(fr)
                dw = [a - b for a, b in zip(w + [z], [z] + w)]
            n = []
            for j in range(o):
                u = fr + j
                a = w[j] if j < o - 1 else 0.0
                b = w[j - 1] if j > 0 else 0.0
                n.append((u * a + (o - u) * b) / (o - 1))
            w = n
        return torch.stack(w[::-1], 2), torch.stack(dw[::-1], 2)

    def intra(self, x):
        """Excluded-pair corrections, bonds, bends: energies per bead, forces, virials."""
        s, P = self.s, self.P
        xs = x.view(P, s.nmol, self.ns, 3)
        f, out = {}, {}
        z = lambda: torch.zeros_like(xs)
        vir = lambda d, g: torch.einsum("pna,pnb->ab", d, g)
        # excluded charged pairs
        q = self.q.view(s.nmol, self.ns)[0]
        g, e, v = z(), 0.0, 0.0
        nodes, wts = np.polynomial.legendre.leggauss(128)
        kmax, al = 15.0 * self.al, self.al
        for i in range(self.ns):
            for j in range(i + 1, self.ns):
                if float(q[i]) == 0.0 or float(q[j]) == 0.0:
                    continue
                d = xs[:, :, i] - xs[:, :, j]
                r = d.norm(dim=2)
                er, der = _erfc(al * r)
                val, dv = -(1.0 - er) / r, al * der / r + (1.0 - er) / (r * r)
                if kmax > self.kcut:
                    for n, w in zip(nodes, wts):
                        k = 0.5 * (n * (kmax - self.kcut) + kmax + self.kcut)
                        c = (kmax - self.kcut) / math.pi * math.exp(-0.25 * k * k / al ** 2) * w
                        if c < 1e-18:
                            continue
                        a = k * r
                        val = val + c * torch.sin(a) / a
                        dv = dv + c * k * (torch.cos(a) - torch.sin(a) / a) / a
                qq = float(q[i] * q[j])
                e = e + (qq * val).sum(1)
                fv = d * (-qq * dv / r)[:, :, None]
                g[:, :, i] += fv
                g[:, :, j] -= fv
                v = v + vir(d, fv)
        f["vecor"], out["vecor"], out["p_ecor"] = g.view_as(x), e, v
        # bonds (O-H1, O-H2)
        g, e, v = z(), 0.0, 0.0
        c, eq = s.bond_c, float(s.bond_eq[0])
        for k in (1, 2):
            d = xs[:, :, 0] - xs[:, :, k]
            r = d.norm(dim=2)
            y = r - eq
            e = e + sum(float(c[m]) * y ** m for m in range(7)).sum(1)
            dv = sum(m * float(c[m]) * y ** (m - 1) for m in range(1, 7))
            fv = d * (-dv / r)[:, :, None]
            g[:, :, 0] += fv
            g[:, :, k] -= fv
            v = v + vir(d, fv)
        f["vbond"], out["vbond"], out["p_bond"] = g.view_as(x), e, v
        # bend H1-O-H2
        g = z()
        d1, d3 = xs[:, :, 1] - xs[:, :, 0], xs[:, :, 2] - xs[:, :, 0]
        r1, r3 = d1.norm(dim=2, keepdim=True), d3.norm(dim=2, keepdim=True)
        co = (d1 * d3).sum(2, keepdim=True) / (r1 * r3)
        si = torch.sqrt(1.0 - co * co)
        ev, dc = self.bend(co, si)
        f1, f3 = -dc * (d3 / (r1 * r3) - d1 * co / (r1 * r1)), -dc * (d1 / (r1 * r3) - d3 * co / (r3 * r3))
        g[:, :, 1] += f1
        g[:, :, 2] += f3
        g[:, :, 0] -= f1 + f3
        f["vbend"], out["vbend"], out["p_bend"] = g.view_as(x), ev[..., 0].sum(1), vir(d1, f1) + vir(d3, f3)
        return out, f

    def bend(self, co, si):
        """V(theta) of the cosine and sine series, and dV/d cos theta."""
        c, s = [float(v) for v in self.s.bend_c], [float(v) for v in self.s.bend_s]
        e = sum(c[m] * co ** m for m in range(7)) + co * sum(s[m] * si ** (m - 1) for m in range(2, 7)) + s[1] * si
        dc = sum(m * c[m] * co ** (m - 1) for m in range(1, 7)) + sum(s[m] * si ** (m - 1) for m in range(2, 7))
        ds = co * sum((m - 1) * s[m] * si ** (m - 2) for m in range(2, 7)) + s[1]
        return e, dc - ds * co / si

    def tail(self, rc):
        n = self.s.nmol
        h = self.heal
        fact = (1.0 / (h * h)) * (1.0 / rc + 1.0 / (rc - h)) + (2.0 / h ** 3) * math.log((rc - h) / rc)
        return -4.0 * math.pi * 4.0 * self.eps * self.sig ** 6 * (n * (n - 1) // 2) * fact / self.V

    def call(self, x, xm=None):
        """The force call at x [P, N, 3]: energies, pressure tensor, forces [P, N, 3]
        (mode forces when asked for), and the per-bead energies."""
        s, P = self.s, self.P
        xm = x.mean(0) if xm is None else xm
        pb, fp, vp = self.pairs(x, xm)
        ib, fi = self.intra(x)
        zero = torch.zeros(P, dtype=x.dtype, device=self.dev)
        rb, fr, vr = (zero, 0.0, 0.0) if self.respa else self.recip(x)
        mean = lambda v: float(v.sum()) / P
        full = not self.respa
        e = dict.fromkeys(E_KEYS, 0.0)
        e["vbond"], e["vbend"] = mean(ib["vbond"]), mean(ib["vbend"])
        qs, qq = float(np.sum(s.q)), float(np.sum(np.asarray(s.q) ** 2))
        e["vself"] = -qq * self.al * self.self_erf / math.sqrt(math.pi)
        e["vbgr"] = -0.5 * qs * qs * math.pi / (self.al ** 2 * self.V)
        f = fp + self.w_tra * (fi["vbond"] + fi["vbend"])
        pv = vp + self.w_tra * (ib["p_bond"] + ib["p_bend"])
        if full:
            e.update(vvdw=mean(pb["vvdw"]), vcoul=mean(pb["vcoul"]), vlong=self.tail(self.rc), vrecip=mean(rb),
                     vecor=mean(ib["vecor"]))
            e["vreal"] = e["vvdw"] + e["vcoul"]
            f, pv = f + fr + fi["vecor"], pv + vr + ib["p_ecor"]
            diag = e["vlong"] * P
        else:
            bead = -(3 * self.nreal // 3) * self.T / water.BOLTZ * P
            diag = bead - bead * self.w_tra + self.tail(min(self.rc, self.rr)) * P * self.w_res
        diag += e["vbgr"] * self.w_tra * P
        e["vintert"] = e["vreal"] + e["vlong"] + e["vrecip"] + e["vself"] + e["vbgr"] + e["vecor"] if full else 0.0
        e["vintrat"] = e["vbond"] + e["vbend"]
        pv = pv + diag * torch.eye(3, dtype=x.dtype, device=self.dev)
        self.bead = {**{k: pb[k] for k in pb}, **{k: ib[k] for k in ("vecor", "vbond", "vbend")}, "vrecip": rb}
        if P > 1:
            f, pv = f / P, pv / P
            d = x - xm
            cor = -torch.einsum("pna,pnb->ab", d, f)
            pv = pv + cor
            if full:
                e["pi_ke_vir"] = 0.5 * (3.0 * self.nreal * self.T / water.BOLTZ + float(torch.trace(cor)))
        if len(s.ghost_atom):
            fm = f.view(P, s.nmol, self.ns, 3).clone()
            site, comp = s.model.ghost
            for k, c in comp:
                fm[:, :, k] += c * fm[:, :, site]
            fm[:, :, site] = 0.0
            f = fm.view_as(f)
        if self.modes:
            u, f = self.to_modes(x) / P, self.to_modes(f)
            f[1:P - 1] *= 2.0
            fk = self.mass * self.T * self.T * P / (2.0 * water.BOLTZ ** 2)
            fk = fk.clone()
            fk[torch.as_tensor(s.ghost_atom.astype(np.int64), device=self.dev)] = 0.0
            lam = torch.as_tensor(_mode_mass(P), device=self.dev)
            lam[0] = 0.0
            k = lam[:, None] * fk[None, :]
            f = f - 2.0 * k[:, :, None] * u
            e["kin_harm"] = float((k * u.square().sum(2)).sum())
            e["pi_ke_prim"] = 1.5 * self.nreal * self.T * P / water.BOLTZ - e["kin_harm"]
        # PINY's tensor order: row b of the column-major 3x3 (symmetric but for the bead correction)
        tot = pv.reshape(-1).cpu().numpy()
        return {"energies": np.array([e[k] for k in E_KEYS]), "pvten": tot, "pvten_tot": tot * full, "nver": None}, f

    def basis(self):
        P = self.P
        b, m = np.arange(P), np.zeros((P, P))
        m[0], m[P - 1] = 1.0, np.where(b % 2, -1.0, 1.0)
        for k in range(1, P // 2):
            m[2 * k - 1], m[2 * k] = np.cos(2 * math.pi * k * b / P), np.sin(2 * math.pi * k * b / P)
        return torch.as_tensor(m, device=self.dev)

    def to_modes(self, x):
        return torch.tensordot(self.basis(), x, dims=([1], [0]))

    def from_modes(self, u):
        w = torch.full((self.P,), 2.0, dtype=u.dtype, device=self.dev)
        w[0] = w[-1] = 1.0
        return torch.tensordot(self.basis() * w[:, None], u, dims=([0], [0]))


def _positions(cfg, dev):
    P, N = cfg.system.pi_beads, cfg.system.natm
    return torch.as_tensor(np.stack([v.reshape(P, N) for v in (cfg.x, cfg.y, cfg.z)], 2), device=dev)


def _device_layout(f):
    """[P, N, 3] as the three site-major arrays of the device forces."""
    return [f[:, :, d].t().contiguous().reshape(-1) for d in range(3)]


def _exact_box(case, cfg):
    ex = _Exact(cfg, respa=case.get("respa", False), modes=case.get("modes", False))
    out, f = ex.call(_positions(cfg, ex.dev))
    return {**out, "forces": _device_layout(f)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        out = [_exact_box(case, c) for c in _batch_configs(case, seed)]
        forces = [o.pop("forces") for o in out]
        return _stacked(out, forces)
    cfg = _config(case, seed)
    if kind == "force":
        return _exact_box(case, cfg)
    if kind == "grad":
        return _exact_grad(cfg)
    vel = np.stack([v.reshape(case["beads"], -1) for v in _velocities(cfg.system, case["beads"], seed)], 2)
    return _exact_nve(cfg, vel, case["steps"]) if kind == "nve" else _exact_pimd(cfg, vel, case["steps"])


def _ghosts(ex, x):
    if ex.s.model.ghost is None:
        return x
    site, comp = ex.s.model.ghost
    xs = x.reshape(ex.P, ex.s.nmol, ex.ns, 3).clone()
    xs[:, :, site] = sum(c * xs[:, :, k] for k, c in comp)
    return xs.view_as(x)


def _exact_nve(cfg, vel, steps):
    ex = _Exact(cfg)
    x, v = _positions(cfg, ex.dev), torch.as_tensor(vel, device=ex.dev)
    dt, im = 0.5 / abi.TIME_CONV, 1.0 / ex.mass[None, :, None]
    out, f = ex.call(x)
    for _ in range(steps):
        v = v + f * im * (dt / 2.0)
        x = _ghosts(ex, x + v * dt)
        out, f = ex.call(x)
        v = v + f * im * (dt / 2.0)
    h = lambda t: t.cpu().numpy()
    return {**out, "kinetic": float(0.5 * (ex.mass[None, :, None] * v * v).sum()), "x": h(x), "v": h(v), "f": h(f)}


def _chain(v, x, Q, kT, kin, dt, nres=4):
    """One Nose-Hoover chain (lists over its links) over a whole step in the
    Suzuki-Yoshida form of three weights; returns the velocity scale."""
    c = 2.0 ** (1.0 / 3.0)
    n, sc = len(v), 1.0
    force = lambda: [(kin - kT[0]) / Q[0]] + [(Q[j] * v[j] * v[j] - kT[j + 1]) / Q[j + 1] for j in range(n - 1)]
    F = force()
    for _ in range(nres):
        for w in (1.0 / (2.0 - c), -c / (2.0 - c), 1.0 / (2.0 - c)):
            h = w * dt / nres
            v[n - 1] = v[n - 1] + F[n - 1] * h / 4
            for j in range(n - 2, -1, -1):
                a = torch.exp(-h / 8 * v[j + 1])
                v[j] = v[j] * a * a + h / 4 * F[j] * a
            a = torch.exp(-h / 2 * v[0])
            sc, kin = sc * a, kin * a * a
            for j in range(n):
                x[j] = x[j] + v[j] * h / 2
            F[0] = (kin - kT[0]) / Q[0]
            for j in range(n - 1):
                a = torch.exp(-h / 8 * v[j + 1])
                v[j] = v[j] * a * a + h / 4 * F[j] * a
                F[j + 1] = (Q[j] * v[j] * v[j] - kT[j + 1]) / Q[j + 1]
            v[n - 1] = v[n - 1] + F[n - 1] * h / 4
    return sc


def _exact_pimd(cfg, vel, steps):
    ex, par = _Exact(cfg, modes=True), abi.nhc_params(gamma_adb=1.0)
    s, P, n, dt = ex.s, ex.P, par.len_nhc, par.dt
    x, v = _positions(cfg, ex.dev), torch.as_tensor(vel, device=ex.dev)
    m = torch.as_tensor(_mode_mass(P), device=ex.dev)[:, None, None] * ex.mass[None, :, None]
    real = torch.ones(ex.N, dtype=torch.bool, device=ex.dev)
    real[torch.as_tensor(s.ghost_atom.astype(np.int64), device=ex.dev)] = False
    kT = ex.T / water.BOLTZ
    tau2 = par.tau_nhc ** 2
    Qc, kc = [tau2 * kT * 3.0 * ex.nreal] + [tau2 * kT] * (n - 1), [3.0 * ex.nreal * kT] + [kT] * (n - 1)
    Qb = [water.BOLTZ ** 2 / P / ex.T ** 2 * kT] * n
    z = lambda: torch.zeros((), dtype=x.dtype, device=ex.dev)
    cv, cx = [z() for _ in range(n)], [z() for _ in range(n)]
    bv = [torch.zeros(P - 1, int(real.sum()), 3, dtype=x.dtype, device=ex.dev) for _ in range(n)]
    bx = [b.clone() for b in bv]

    def chains():
        kin = (m[0][real] * v[0][real] ** 2).sum()
        v[0][real] = v[0][real] * _chain(cv, cx, Qc, kc, kin, dt)
        w = v[1:, real]
        v[1:, real] = w * _chain(bv, bx, Qb, [kT] * n, m[1:, real] * w * w, dt)

    out, f = ex.call(x)
    for _ in range(steps):
        chains()
        v = v + f * (dt / 2.0) / m
        u = ex.to_modes(x) / P + v * dt
        x = _ghosts(ex, ex.from_modes(u))
        out, f = ex.call(x, u[0])
        v = v + f * (dt / 2.0) / m
        chains()
    ke = float(0.5 * (m * v * v).sum())
    en = sum(float(0.5 * Q * a * a + k * b) for Q, k, a, b in zip(Qc, kc, cv, cx))
    en += sum(float((0.5 * Q * a * a + kT * b).sum()) for Q, a, b in zip(Qb, bv, bx))
    pot = sum(out["energies"][E_KEYS.index(k)] for k in ("vintert", "vintrat", "kin_harm"))
    # chain state: the centroid chain, then [mode][site][direction][v.., x..]
    st = torch.zeros(P - 1, ex.N, 3, 2 * n, dtype=x.dtype, device=ex.dev)
    st[:, real] = torch.stack(bv + bx, 3)
    st = torch.cat([torch.stack(cv + cx), st.reshape(-1)]).cpu().numpy()
    h = lambda t: t.cpu().numpy()
    return {**out, "econs": np.array([ke, en, pot, ke + en + pot]), "x": h(x), "v": h(v), "f": h(f), "chains": st}


def _exact_grad(cfg):
    ex = _Exact(cfg)
    mod = cfg.system.model
    x = _positions(cfg, ex.dev)
    out, f = ex.call(x)
    e = dict(zip(E_KEYS, out["energies"]))
    b = ex.bead
    const = e["vlong"] + e["vself"] + e["vbgr"]
    energy = b["vcoul"] + b["vvdw"] + b["vrecip"] + b["vecor"] + b["vbond"] + b["vbend"] + const
    tot = {k: float(v.sum()) for k, v in b.items()}
    P, q_h = ex.P, mod.charges[mod.sites.index("H")]
    d = lambda v: torch.tensor(float(v), dtype=torch.float64)
    g = {"q_h": d(2.0 * (tot["vcoul"] + tot["vrecip"] + tot["vecor"] + P * (e["vself"] + e["vbgr"])) / q_h),
         "epsilon": d((tot["vvdw"] + P * e["vlong"]) / mod.lj_eps_kcal),
         "sigma": d((12.0 * tot["a12"] - 6.0 * tot["a6"] + 6.0 * P * e["vlong"]) / mod.lj_sig)}
    # bonds and bends: the model's own functions of its parameters
    xs = x.view(P, ex.s.nmol, ex.ns, 3)
    d1, d2 = xs[:, :, 1] - xs[:, :, 0], xs[:, :, 2] - xs[:, :, 0]
    r1, r2 = d1.norm(dim=2), d2.norm(dim=2)
    kcal = 1.0 / water.KB_KCAL / water.BOLTZ
    p = {k: v.to(ex.dev).requires_grad_(True) for k, v in autograd.water_params(mod).items()}
    yb = torch.stack([r1, r2]) * water.BOHR - p["r0"]
    if "morse_d" in p:
        a = p["morse_a"] * yb
        eb = p["morse_d"] * kcal * (a ** 2 - a ** 3 + 7.0 / 12.0 * a ** 4 - a ** 5 / 4.0 + 31.0 / 360.0 * a ** 6)
    else:
        eb = 0.5 * p["bond_k"] * kcal * yb ** 2
    co = (d1 * d2).sum(2) / (r1 * r2)
    # 1/2 k (theta - theta0)^2 as the series in y = sin(theta - theta0)^2
    th = torch.acos(co) - p["theta0"] * (math.pi / 180.0)
    y = torch.sin(th) ** 2
    ea = 0.5 * p["k_theta"] * kcal * (y + y ** 2 / 3.0 + 8.0 / 45.0 * y ** 3)
    (eb.sum() + ea.sum()).backward()
    g.update({k: p[k].grad.cpu() for k in p if k not in g})
    return {"energy": energy, "x": -(f * P), **{k: g[k] for k in p}}
