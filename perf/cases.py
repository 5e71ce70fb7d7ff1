"""The work a user of this library has it do, as cases that can be timed.

Every case goes through the public entry points: the device-resident engine
(molmodel_amd.engine.Engine over include/molmodel_amd.h) or the
reference-named drop-ins (include/molmodel_amd_ref.h).  Kinds:

  md      a block of rigid-water MD steps from one frame to the next (50 fs,
          short enough that rounding has not grown into another trajectory)
          (Engine.md_run over replayed graphs), then the frame is read;
  force   one force evaluation per call on coordinates the caller holds
          (set_positions, compute, forces, energies[, virial]): a minimiser
          or an outer MD loop that keeps its own integrator ("near": each
          call moves the sites a little), or a stored trajectory evaluated
          again ("far": each call brings an unrelated frame, so the
          neighbour list is rebuilt);
  grad    the parameter gradients of energy and force-matching loss (the
          backward direction);
  remd    one replica-exchange interval of a batch of systems;
  dropin  RSpaceEwald plus p3m_field or kspace_field, called as ElecLJ calls
          them, on host arrays and the caller's neighbour rows.

Systems are rigid three-site water boxes at liquid density, with or without
ions, from the repository's generator; sizes run from its smallest workload
(216 waters) to its benchmark's (32 768 waters, 98 304 atoms).  Odd sizes
take waters out of a box at random.

Pair and mesh arithmetic of the library are FP32 with FP64 sums, so what
comes back has FP32 precision; run() hands it on as float32, the form a
trajectory file or a model takes.  The Ewald sums of the drop-in are FP64
throughout and stay float64.

exact() restates the same quantities in FP64 with torch: erfc itself in
place of the library's table, the same P3M (assignment, influence function,
differentiation) or Ewald sum, the same constraints and integrator.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from molmodel_amd import engine as E
from molmodel_amd import waterbox as W

SPACING = 3.1067          # A between lattice waters at liquid density
DT = 0.001                # ps
P = C.c_void_p


# ------------------------------------------------------------------ cases

def _case(kind, nwater, boxl, **kw):
    c = dict(kind=kind, nwater=nwater, nion=0, boxl=boxl, rc=10.0, eta=0.32, kmode=1, kc=7.0,
             nx=0, ny=0, nz=0, order=5, ik=0, steps=0, virial=0, frames="", nrep=0, tuned=0)
    c.update(kw)
    return c


def listed():
    mesh = lambda n: dict(nx=n, ny=n, nz=n)
    small = dict(rc=9.0, eta=0.35, kmode=0)
    return [
        # the smallest MD: launches and latency are all there is
        dict(name="md_216_ewald", **_case("md", 216, 18.64, steps=50, **small)),
        # solution of ions: one-site groups beside the waters
        dict(name="md_960_ions_ewald", **_case("md", 960, 31.4, nion=40, kmode=0, steps=50)),
        # an ordinary solvated-protein-sized box
        dict(name="md_4096_p3m48", **_case("md", 4096, 49.7, steps=50, **mesh(48))),
        # the benchmark's box
        dict(name="md_32768_p3m64", **_case("md", 32768, 99.4, steps=50, **mesh(64))),
        # field formed on the mesh (momentum-conserving MD), a box that is no
        # full lattice, a mesh with every radix
        dict(name="md_2900_ik45", **_case("md", 2900, 15 * SPACING, steps=50, ik=1, order=4,
                                          nx=45, ny=42, nz=48)),
        # an outer program's MD loop or minimiser at the benchmark's size
        dict(name="force_32768_near", **_case("force", 32768, 99.4, frames="near", **mesh(64))),
        # energies, forces and pressure of stored frames
        dict(name="force_4096_far", **_case("force", 4096, 49.7, frames="far", virial=1,
                                            **mesh(48))),
        # a small ragged box, high assignment order, one evaluation at a time
        dict(name="force_500_near", **_case("force", 500, 8 * SPACING, nion=8, frames="near",
                                            order=6, nx=27, ny=30, nz=32)),
        # force-field fitting: small box with ions, and an ordinary P3M box
        dict(name="grad_960_ions_ewald", **_case("grad", 960, 31.4, nion=40, kmode=0)),
        dict(name="grad_4096_p3m48", **_case("grad", 4096, 49.7, **mesh(48))),
        # replica exchange over 48 systems of three sizes, in the shape the
        # autotuner chooses for it
        dict(name="remd_48", **_case("remd", 0, 0.0, nrep=16, steps=50, tuned=1)),
        # the reference's own functions relinked
        dict(name="dropin_4096_p3m48", **_case("dropin", 4096, 49.7, **mesh(48))),
    ]


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["md", "md", "md", "force", "force", "grad", "remd", "dropin"])
    if kind == "remd":
        return _case("remd", 0, 0.0, nrep=rng.randint(2, 16), steps=rng.randint(10, 50),
                     tuned=rng.randint(0, 1))
    most = {"md": 32768, "force": 32768, "grad": 4096, "dropin": 4096}[kind]
    n = int(round(math.exp(rng.uniform(math.log(216), math.log(most)))))
    kw = dict(nion=2 * rng.randint(1, 20) if n > 300 and rng.random() < 0.4 else 0)
    boxl = _side(n + kw["nion"]) * SPACING
    kw["rc"] = 9.0 if boxl < 20.5 else 10.0
    if n < 1500 and rng.random() < 0.5:
        kw.update(kmode=0, eta=0.35 if kw["rc"] == 9.0 else 0.32, kc=rng.choice([6.0, 7.0, 7.5]))
    else:
        kw.update(eta=rng.uniform(0.28, 0.36), order=rng.choice([3, 4, 5, 5, 6]),
                  ik=int(rng.random() < 0.25))
        for k in ("nx", "ny", "nz"):
            kw[k] = min(W.smooth_mesh_size(round(boxl * rng.uniform(0.65, 1.1))), 100)
        if rng.random() < 0.5:
            kw.update(ny=kw["nx"], nz=kw["nx"])
    if kind == "md":
        kw["steps"] = rng.randint(10, 50)
    if kind == "force":
        kw.update(frames=rng.choice(["near", "near", "far"]), virial=rng.randint(0, 1))
    return _case(kind, n, boxl, **kw)


# ------------------------------------------------------- systems and inputs

def _side(n):
    return math.ceil(n ** (1 / 3) - 1e-9)


def _system(case, seed):
    """nwater waters and nion ions (half Na+, half Cl-), each in a place of
    its own on the generator's lattice, the places that are left empty."""
    n, ni, L = case["nwater"], case["nion"], case["boxl"]
    side = _side(n + ni)
    s = W.water_box(side, L, seed=seed + 1)
    if n < side ** 3:
        rng = np.random.default_rng(seed)
        place = rng.permutation(side ** 3)
        at = s.r[3 * place[n:n + ni]]
        s = W.subset(s, np.sort(place[:n]))
    if ni:
        kinds = [W.IONS["Na"]] * (ni // 2) + [W.IONS["Cl"]] * (ni - ni // 2)
        of = lambda k: np.array([x[k] for x in kinds])
        mass = W.g_mol_to_mass_unit(of("m"))
        vi = rng.normal(size=(ni, 3)) * np.sqrt(W.K_to_kcal_mol(300.0) / mass)[:, None]
        first = s.nsite + np.arange(ni, dtype=np.int32)
        s.r, s.v = np.concatenate([s.r, at]), np.concatenate([s.v, vi])
        s.q = np.concatenate([s.q, W.e_to_charge_unit(of("q"))])
        s.sig, s.eps = np.concatenate([s.sig, of("sig")]), np.concatenate([s.eps, of("eps")])
        s.mass = np.concatenate([s.mass, mass])
        s.site_mask = np.concatenate([s.site_mask, np.full(ni, 3, dtype=np.int32)])
        s.group = np.concatenate([s.group, np.stack([first, first + 1], 1)]).astype(np.int32)
        s.nion = ni
    p = dict(rc=case["rc"], smoothing_width=1.0, eta=case["eta"], kmode=case["kmode"],
             kc=case["kc"], mesh=(case["nx"], case["ny"], case["nz"]), order=case["order"],
             ik=case["ik"], nalias=2, include_lj_correction=1,
             skin=W.default_skin(case["rc"], L))
    return s, p


def _frames(case, s, seed):
    """Coordinates of successive calls: small rigid moves of every molecule,
    or unrelated frames."""
    if case["frames"] == "far":
        return [s.r, _system(case, seed + 500_000)[0].r]
    size = np.diff(s.group, axis=1)[:, 0]
    move = lambda k: np.random.default_rng(seed + k).normal(0.0, 0.03, (s.ngroup, 3))
    return [s.r] + [s.r + np.repeat(move(k), size, axis=0) for k in (1, 2, 3)]


def _remd(case, seed):
    def ks(boxl, nsite, rc):
        c = E.tune_kspace(boxl, nsite, rc, 1e-4)
        return {k: v for k, v in c.items() if k in ("eta", "kmode", "kc", "mesh", "order")}

    # the autotuner's choice for this batch on one MI355X
    shape = dict(cell_groups=1, pair_slots=4, spread_block=4, graph_steps=20, spread_halo=1)
    return W.remd_batch(nrep=case["nrep"], seed=seed + 7, kspace=ks) + \
        (shape if case["tuned"] else None,)


def _f_ref(s, seed):
    """Reference forces of a fit: the size of liquid water's, from elsewhere."""
    return np.random.default_rng(seed + 9).normal(0.0, 15.0, s.r.shape)


def _lib():
    L = E.lib()
    I, D = C.c_int, C.c_double
    L.PairBinary_new.restype = P
    L.PairBinary_new.argtypes = [I]
    L.PairBinary_quick_add.argtypes = [P, I, I]
    L.PairBinary_init.argtypes = [P]
    L.RSpaceEwald.restype = None
    L.RSpaceEwald.argtypes = [I, I, P, P, I, P, P, P, P, P, D, D, P, P, P, P, D, P, P, P, P, I,
                              P, P, P, D, D]
    L.p3m_new.restype = P
    L.p3m_new.argtypes = [I, P, D, I, I, I, P]
    L.p3m_init.argtypes = [P, D, P]
    L.p3m_field.argtypes = [P, P, P, P, P]
    L.p3m_delete.argtypes = [P]
    L.kspace_new.restype = P
    L.kspace_new.argtypes = [D, I]
    L.kspace_field.argtypes = [P, P, P, P, D, D, P, P]
    L.kspace_delete.argtypes = [P]
    L.PairBinary_delete.argtypes = [P]
    return L


class _Dropins:
    """What ElecLJ holds between force evaluations: neighbour rows, excluded
    pairs and the k-space or P3M handle."""

    def __init__(self, case, s, p):
        L = self.L = _lib()
        self.s, self.p = s, p
        self.latv = np.diag([s.boxl] * 3).astype(np.float64).reshape(-1)
        self.r = np.ascontiguousarray(s.r)
        self.group = np.ascontiguousarray(s.group)
        self.mask = np.ascontiguousarray(s.site_mask)
        # neighbour rows as the reference's list holds them
        e = E.Engine(s, p)
        e.set_positions(s.r)
        pairs = e.nl_pairs(0)
        e.close()
        pairs = pairs[np.lexsort((pairs[:, 1], pairs[:, 0]))]
        self.nn = np.bincount(pairs[:, 0], minlength=s.ngroup).astype(np.int32)
        self.cols = np.ascontiguousarray(pairs[:, 1], dtype=np.int32)
        start = np.concatenate([[0], np.cumsum(self.nn)[:-1]])
        self.rows = (self.cols.ctypes.data + 4 * start).astype(np.uint64)
        self.excl = L.PairBinary_new(s.nsite)
        for a, b in s.excl.tolist():
            L.PairBinary_quick_add(self.excl, *((b, a) if ((a + b) % 2) ^ (a < b) else (a, b)))
        L.PairBinary_init(self.excl)
        self.gexcl = L.PairBinary_new(s.ngroup)
        L.PairBinary_init(self.gexcl)
        self.mesh = None
        if p["kmode"] == 1:
            ng, chi = np.zeros(3, dtype=np.int32), C.c_double()
            self.k = L.p3m_new(s.nsite, _p(self.latv), s.boxl / case["nx"], p["nalias"], p["ik"],
                               p["order"], _p(ng))
            L.p3m_init(self.k, p["eta"], C.byref(chi))
            self.mesh = tuple(int(x) for x in ng)
        else:
            self.k = L.kspace_new(p["kc"], s.nsite)

    def __del__(self):
        (self.L.p3m_delete if self.p["kmode"] == 1 else self.L.kspace_delete)(self.k)
        self.L.PairBinary_delete(self.excl)
        self.L.PairBinary_delete(self.gexcl)

    def run(self):
        s, p, L = self.s, self.p, self.L
        phi, ev, ljf = np.zeros(s.nsite), np.zeros((s.nsite, 3)), np.zeros((s.nsite, 3))
        lje = np.zeros(1)
        L.RSpaceEwald(s.nsite, s.ngroup, _p(self.group), _p(self.r), 1, _p(self.latv),
                      _p(self.rows), _p(self.nn), self.gexcl, self.excl,
                      (p["rc"] - p["smoothing_width"]) ** 2, p["rc"] ** 2, _p(self.mask),
                      _p(s.q), _p(phi), _p(ev), p["eta"], None, None, _p(s.sig), _p(s.eps), 0,
                      _p(lje), _p(ljf), None, 1.0, 1.0)
        kphi, kev = np.zeros(s.nsite), np.zeros((s.nsite, 3))
        if p["kmode"] == 1:
            L.p3m_field(self.k, _p(self.r), _p(s.q), _p(kphi), _p(kev))
            kphi, kev = kphi.astype(np.float32), kev.astype(np.float32)
        else:
            rl = 2 * math.pi / s.boxl * np.diag([1.0] * 3)
            L.kspace_field(self.k, _p(self.r), _p(s.q), _p(rl), s.boxl ** 3, p["eta"], _p(kphi),
                           _p(kev))
        f = np.float32
        return dict(phi=phi.astype(f), evec=ev.astype(f), lj_force=ljf.astype(f),
                    lj_energy=lje.astype(f), kphi=kphi, kevec=kev)


def _p(a):
    return a.ctypes.data_as(P)


class _State:
    pass


def prepare(case, seed):
    st = _State()
    st.case, st.call = case, 0
    kind = case["kind"]
    if kind == "remd":
        systems, params, kT, ladders, shape = _remd(case, seed)
        e = st.e = E.Engine(systems, params, shape=shape)
        e.set_positions(np.concatenate([s.r for s in systems]))
        e.set_velocities(np.concatenate([s.v for s in systems]))
        e.md_setup(dt=DT)
        e.remd_setup(ladders, kT, seed=seed + 11)
        return st
    s, p = _system(case, seed)
    if kind == "dropin":
        st.d = _Dropins(case, s, p)
        return st
    e = st.e = E.Engine(s, p)
    if kind == "md":
        e.set_positions(s.r)
        e.set_velocities(s.v)
        e.md_setup(dt=DT)
    elif kind == "force":
        st.frames = [np.ascontiguousarray(r) for r in _frames(case, s, seed)]
    elif kind == "grad":
        e.set_positions(s.r)
        st.f_ref = _f_ref(s, seed)
    return st


# the documented energy slots: elec, lj, tail, total, kinetic, kspace
NSLOT = 6


def run(st):
    case, f = st.case, np.float32
    kind = case["kind"]
    if kind == "md":
        e = st.e
        e.md_run(case["steps"])
        return dict(r=e.positions().astype(f), v=e.velocities().astype(f),
                    f=e.forces().astype(f), energies=e.energies()[:, :NSLOT].astype(f))
    if kind == "force":
        e = st.e
        e.set_positions(st.frames[st.call % len(st.frames)])
        st.call += 1
        e.compute(virial=bool(case["virial"]))
        out = dict(f=e.forces().astype(f), energies=e.energies()[:, :NSLOT].astype(f))
        if case["virial"]:
            out["virial"] = e.virial().astype(f)
        return out
    if kind == "grad":
        g = st.e.param_gradients(0, f_ref=st.f_ref)
        return dict(dE=g["dE"].astype(f), dL=g["dL"].astype(f), loss=np.float32(g["loss"]))
    if kind == "remd":
        e = st.e
        e.remd_run(1, case["steps"])
        _, cfg = e.remd_stats()
        return dict(r=e.positions().astype(f), v=e.velocities().astype(f),
                    energies=e.energies()[:, :NSLOT].astype(f), config=cfg)
    return st.d.run()


# ------------------------------------------------------------------- work

def work(case):
    """Per force evaluation: each unordered site pair once (39 operations a
    charged pair, 32 an LJ pair, 14 a group pair), order^3 weights per site
    to and from the mesh and two transforms, or sine and cosine sums over
    the wave vectors; state read and written once."""
    if case["kind"] == "remd":
        sizes = [(216, 18.64, 9.0, 0), (512, 24.86, 10.0, 30), (1000, 31.07, 10.0, 36)]
        tot = [0.0, 0.0]
        for n, L, rc, m in sizes:
            c = _case("md", n, L, rc=rc, kmode=1 if m else 0, nx=m, ny=m, nz=m, order=6,
                      steps=case["steps"] + 1)
            w = work(c)
            tot[0] += case["nrep"] * w["bytes"]
            tot[1] += case["nrep"] * w["flops"]
        return dict(bytes=tot[0], flops=tot[1])
    n, L, rc = case["nwater"], case["boxl"], case["rc"]
    ns = 3 * n + case["nion"]
    g = 0.5 * n * n * 4 / 3 * math.pi * rc ** 3 / L ** 3
    flops, byts = g * (14 + 9 * 39 + 32), 0.0
    if case["kmode"] == 1:
        m = case["nx"] * case["ny"] * case["nz"]
        c = 4 if case["ik"] else 1
        flops += ns * case["order"] ** 3 * (2 + 8) + (1 + c) * 2.5 * m * math.log2(m)
        byts += 4.0 * m * (1 + c)
    else:
        flops += ns * 2 / 3 * math.pi * case["kc"] ** 3 * 2 * 20
    kind = case["kind"]
    if kind == "md":   # positions, velocities, forces in and out
        return dict(bytes=case["steps"] * (byts + 2 * 72.0 * ns),
                    flops=case["steps"] * (flops + 300.0 * n))
    if kind == "force":
        return dict(bytes=byts + 48.0 * ns, flops=flops)
    if kind == "grad":   # forward and backward, each pair again
        return dict(bytes=2 * byts + 100.0 * ns, flops=3 * flops)
    return dict(bytes=byts + 4.0 * 80 * n + 136.0 * ns, flops=flops)


# ------------------------------------------------------- the FP64 statement

class _Exact:
    """Forces, energies, virial of one system in FP64."""

    def __init__(self, case, s, p, mesh=None):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.case, self.s, self.p, self.L = case, s, p, s.boxl
        t = lambda a, d=torch.float64: torch.as_tensor(np.asarray(a), dtype=d, device=self.dev)
        self.q, self.sig, self.eps, self.m = t(s.q), t(s.sig), t(s.eps), t(s.mass)
        i64 = torch.int64
        self.g0 = t(s.group[:, 0], i64)
        self.ns = t(s.group[:, 1] - s.group[:, 0], i64)
        self.mask = t(s.site_mask, i64)
        self.excl = t(s.excl, i64).reshape(-1, 2)
        self.water = torch.nonzero(self.ns == 3)[:, 0]
        self.mesh = mesh or p["mesh"]
        self.pairs = None
        self._recip()

    # -- reciprocal space
    def _recip(self):
        p, L, dev = self.p, self.L, self.dev
        V, eta = L ** 3, p["eta"]
        if p["kmode"] == 0:
            kc = p["kc"]
            m = int(math.floor(kc))
            a = torch.arange(-m, m + 1, device=dev, dtype=torch.float64)
            n = torch.stack(torch.meshgrid(a, a, a, indexing="ij"), -1).reshape(-1, 3)
            half = (n[:, 0] > 0) | ((n[:, 0] == 0) & ((n[:, 1] > 0) |
                                                    ((n[:, 1] == 0) & (n[:, 2] > 0))))
            n = n[half & ((n * n).sum(1) <= kc * kc + 1e-8)]
            self.k = n * (2 * math.pi / L)
            k2 = (self.k ** 2).sum(1)
            self.a = 4 * math.pi / V * torch.exp(-k2 / (4 * eta * eta)) / k2
            return
        nx, ny, nz = self.mesh
        na, order = p["nalias"], p["order"]
        idx = lambda n: torch.where(torch.arange(n, device=dev) > n // 2,
                                    torch.arange(n, device=dev) - n,
                                    torch.arange(n, device=dev)).to(torch.float64)
        j = [idx(nx), idx(ny), torch.arange(nz // 2 + 1, device=dev, dtype=torch.float64)]
        n3 = (nx, ny, nz)
        sh = [(-1, 1, 1), (1, -1, 1), (1, 1, -1)]
        self.kk = [(2 * math.pi / L * j[d]).reshape(sh[d]) for d in range(3)]
        num = d1 = d2 = 0
        for ax in range(-na, na + 1):
            for ay in range(-na, na + 1):
                for az in range(-na, na + 1):
                    al = (ax, ay, az)
                    kp = [(2 * math.pi / L * (j[d] + al[d] * n3[d])).reshape(sh[d])
                          for d in range(3)]
                    u = [torch.special.sinc(j[d] / n3[d] + al[d]).pow(2 * order).reshape(sh[d])
                         for d in range(3)]
                    u2 = u[0] * u[1] * u[2]
                    k2 = kp[0] ** 2 + kp[1] ** 2 + kp[2] ** 2
                    ok = k2 > 0
                    gg = torch.where(ok, 4 * math.pi / torch.where(ok, k2, 1.0) *
                                     torch.exp(-k2 / (4 * eta * eta)), 0.0)
                    u2 = torch.where(ok, u2, 0.0)
                    if p["ik"]:
                        num = num + gg * u2 * sum(a * b for a, b in zip(self.kk, kp))
                    else:
                        num = num + gg * u2 * k2
                        d2 = d2 + u2 * k2
                    d1 = d1 + u2
        k2 = self.kk[0] ** 2 + self.kk[1] ** 2 + self.kk[2] ** 2
        den = d1 * d1 * k2 if p["ik"] else d1 * d2
        g = num / torch.where(k2 > 0, den, 1.0) / V
        self.G = torch.where(k2 > 0, g, 0.0)
        self.mult = torch.full((nz // 2 + 1,), 2.0, device=dev, dtype=torch.float64)
        self.mult[0] = 1.0
        if nz % 2 == 0:
            self.mult[-1] = 1.0

    def _weights(self, x, n):
        """Base index and the order's weights (and derivatives) along one axis."""
        o = self.p["order"]
        s = x * (n / self.L)
        if o & 1:
            j = torch.floor(s + 0.5)
            f = s - j
        else:
            j = torch.floor(s)
            f = s - j - 0.5
        u = f + 0.5
        m = [torch.ones_like(u)] + [torch.zeros_like(u)] * o
        for k in range(2, o + 1):
            if k == o:
                low = list(m)
            m = [((u + i) * m[i] + (k - u - i) * (m[i - 1] if i else 0.0)) / (k - 1)
                 for i in range(k)] + [torch.zeros_like(u)] * (o + 1 - k)
        w = torch.stack([m[o - 1 - i] for i in range(o)], -1)
        dw = torch.stack([(low[o - 1 - i] if o - 1 - i < o - 1 else 0 * u) -
                          (low[o - 2 - i] if o - 2 - i >= 0 else 0 * u)
                          for i in range(o)], -1) * (n / self.L)
        at = (j.to(torch.int64)[:, None] - ((o + 1) // 2 - 1) +
              torch.arange(o, device=self.dev)) % n
        return at, w, dw

    def _ifft(self, c):
        nx, ny, nz = self.mesh
        y = torch.fft.ifftn(c, dim=(0, 1)) * (nx * ny)
        keep = torch.ones(nz // 2 + 1, device=self.dev, dtype=torch.float64)
        keep[0] = 0
        if nz % 2 == 0:
            keep[-1] = 0
        y = torch.complex(y.real, y.imag * keep)
        return torch.fft.irfft(y, n=nz, dim=2) * nz

    def recip(self, r, q):
        """phi, E per site; energy, virial of the mesh or k sum."""
        p, eta = self.p, self.p["eta"]
        c4 = 0.25 / (eta * eta)
        if p["kmode"] == 0:
            phi, ev = [], []
            arg = r @ self.k.T
            sn, cs = torch.sin(arg), torch.cos(arg)
            S, Cc = q @ sn, q @ cs
            phi = (sn @ (2 * self.a * S)) + (cs @ (2 * self.a * Cc))
            t = 2 * self.a * (sn * Cc - cs * S)
            ev = t @ self.k
            ek = self.a * (S * S + Cc * Cc)
            k2 = (self.k ** 2).sum(1)
            w = torch.eye(3, device=self.dev, dtype=torch.float64) * ek.sum() - \
                (self.k * (2 * ek * (1 / k2 + c4))[:, None]).T @ self.k
            return phi, ev, ek.sum(), w
        nx, ny, nz = self.mesh
        ax, wx, dx = self._weights(r[:, 0], nx)
        ay, wy, dy = self._weights(r[:, 1], ny)
        az, wz, dz = self._weights(r[:, 2], nz)
        at = ((ax[:, :, None, None] * ny + ay[:, None, :, None]) * nz +
              az[:, None, None, :]).reshape(-1)
        three = lambda a, b, c: (a[:, :, None, None] * b[:, None, :, None] * c[:, None, None, :])
        w0 = three(wx, wy, wz)
        n = r.shape[0]
        rho = torch.zeros(nx * ny * nz, device=self.dev, dtype=torch.float64)
        rho = rho.index_add(0, at, (q[:, None, None, None] * w0).reshape(-1)).reshape(nx, ny, nz)
        rk = torch.fft.fft2(torch.fft.rfft(rho, dim=2), dim=(0, 1))
        pk = self.G * rk
        ek = 0.5 * self.mult * self.G * (rk.real ** 2 + rk.imag ** 2)
        k2 = self.kk[0] ** 2 + self.kk[1] ** 2 + self.kk[2] ** 2
        f = 2 * (1 / torch.where(k2 > 0, k2, 1.0) + c4) * ek
        w = torch.stack([torch.stack([(f * self.kk[a] * self.kk[b]).sum() for b in range(3)])
                         for a in range(3)])
        w = torch.eye(3, device=self.dev, dtype=torch.float64) * ek.sum() - w
        take = lambda mesh, wt: (mesh.reshape(-1)[at].reshape(n, -1) * wt.reshape(n, -1)).sum(1)
        ph = self._ifft(pk)
        phi = take(ph, w0)
        if p["ik"]:
            ev = torch.stack([take(self._ifft(torch.complex(self.kk[a] * pk.imag,
                                                            -self.kk[a] * pk.real)), w0)
                              for a in range(3)], 1)
        else:
            ev = -torch.stack([take(ph, three(dx, wy, wz)), take(ph, three(wx, dy, wz)),
                               take(ph, three(wx, wy, dz))], 1)
        return phi, ev, ek.sum(), w

    # -- real space
    def find_pairs(self, r, margin):
        x, L = r[self.g0], self.L
        c2 = (self.p["rc"] + margin) ** 2
        out = []
        for a in range(0, x.shape[0], 2048):
            d2 = 0
            for c in range(3):
                d = x[a:a + 2048, None, c] - x[None, :, c]
                d = d - L * torch.round(d / L)
                d2 = d2 + d * d
            i, j = torch.nonzero(d2 <= c2, as_tuple=True)
            i = i + a
            out.append(torch.stack([i[i < j], j[i < j]]))
        self.pairs = torch.cat(out, 1)

    def rspace(self, r, q, sig, eps):
        """phi, field, LJ force, LJ energy, virial of the pairs in the cutoff
        and of the excluded pairs, and the switching force's share."""
        p, L = self.p, self.L
        rhi2, rlo2 = p["rc"] ** 2, (p["rc"] - p["smoothing_width"]) ** 2
        eta = p["eta"]
        N = r.shape[0]
        i, j = self.pairs
        a, b = self.g0[i], self.g0[j]
        D0 = r[a] - r[b]
        shift = -L * torch.floor(D0 / L + 0.5)
        D = D0 + shift
        r2 = (D * D).sum(1)
        on = r2 <= rhi2
        i, j, a, b, D, shift, r2 = i[on], j[on], a[on], b[on], D[on], shift[on], r2[on]
        z = ((r2 - rlo2) / (rhi2 - rlo2)).clamp(min=0)
        sm = ((-6 * z + 15) * z - 10) * z ** 3 + 1
        dsm = ((60 * z - 120) * z + 60) * z * z / (rhi2 - rlo2)
        zero = lambda *s: torch.zeros(*s, device=self.dev, dtype=torch.float64)
        phi, ev, lj, smf = zero(N), zero(N, 3), zero(N, 3), zero(N, 3)
        w, ulj, tmp = zero(3, 3), zero(()), zero(r2.shape[0])
        ns = self.ns
        for k in range(3):
            for l in range(3):
                ok = (ns[i] > k) & (ns[j] > l)
                if not bool(ok.any()):
                    continue
                x = torch.nonzero(ok)[:, 0]
                u, v = a[x] + k, b[x] + l
                d = r[u] - r[v] + shift[x]
                d2 = (d * d).sum(1)
                m = self.mask[u] & self.mask[v]
                hq = (m & 1).to(torch.float64)
                rm = torch.sqrt(d2)
                b0 = torch.erfc(eta * rm) / rm * hq
                b1 = (b0 + hq * eta * (2 / math.sqrt(math.pi)) * torch.exp(-eta * eta * d2)) / d2
                s0 = sm[x]
                phi = phi.index_add(0, u, q[v] * b0 * s0).index_add(0, v, q[u] * b0 * s0)
                g = (b1 * s0)[:, None] * d
                ev = ev.index_add(0, u, q[v][:, None] * g).index_add(0, v, -q[u][:, None] * g)
                t = q[u] * q[v] * b0
                f = (q[u] * q[v])[:, None] * g
                y = torch.nonzero(m & 2)[:, 0]
                if y.numel():
                    uu, vv, dd = u[y], v[y], d[y]
                    s6 = (0.5 * (sig[uu] + sig[vv])) ** 6
                    bb = 4 * torch.sqrt(eps[uu] * eps[vv]) * s6
                    i6 = 1 / d2[y] ** 3
                    en = bb * s6 * i6 * i6 - bb * i6
                    fl = ((12 * bb * s6 * i6 * i6 - 6 * bb * i6) / d2[y] * s0[y])[:, None] * dd
                    ulj = ulj + (en * s0[y]).sum()
                    lj = lj.index_add(0, uu, fl).index_add(0, vv, -fl)
                    f = f.index_add(0, y, fl)
                    t = t.index_add(0, y, en)
                w = w + d.T @ f
                tmp = tmp.index_add(0, x, t)
        fs = (dsm * tmp)[:, None] * D
        smf = smf.index_add(0, a, fs).index_add(0, b, -fs)
        w = w + D.T @ fs
        if self.excl.numel():
            u, v = self.excl[:, 0], self.excl[:, 1]
            d = r[u] - r[v]
            d = d - L * torch.floor(d / L + 0.5)
            d2 = (d * d).sum(1)
            rm = torch.sqrt(d2)
            b0 = -torch.erf(eta * rm) / rm
            b1 = (b0 + eta * (2 / math.sqrt(math.pi)) * torch.exp(-eta * eta * d2)) / d2
            phi = phi.index_add(0, u, q[v] * b0).index_add(0, v, q[u] * b0)
            g = b1[:, None] * d
            ev = ev.index_add(0, u, q[v][:, None] * g).index_add(0, v, -q[u][:, None] * g)
            w = w + d.T @ ((q[u] * q[v])[:, None] * g)
        return phi, ev, lj + smf, ulj, w

    def tail(self, sig, eps):
        rhi, rlo, V = self.p["rc"], self.p["rc"] - self.p["smoothing_width"], self.L ** 3
        A = B = 0
        lj = torch.nonzero(self.mask & 2)[:, 0]
        key = torch.stack([self.sig[lj], self.eps[lj]], 1)
        _, inv, cnt = torch.unique(key, dim=0, return_inverse=True, return_counts=True)
        kinds = [(int(lj[torch.nonzero(inv == c)[0, 0]]), int(n)) for c, n in enumerate(cnt)]
        for x, nx in kinds:
            for y, ny in kinds:
                s6 = (0.5 * (sig[x] + sig[y])) ** 6
                bb = 4 * torch.sqrt(eps[x] * eps[y]) * nx * ny * s6
                A, B = A + bb * s6, B - bb
        w = (rhi - rlo) / (63 * rhi ** 3 * rlo ** 9 * (rhi + rlo) ** 5)
        ca = 1 / (9 * rlo ** 9) - w * (7 * rhi ** 7 + 42 * rhi ** 6 * rlo +
                                       112 * rhi ** 5 * rlo ** 2 + 182 * rhi ** 4 * rlo ** 3 +
                                       217 * rhi ** 3 * rlo ** 4 + 224 * rhi ** 2 * rlo ** 5 +
                                       192 * rhi * rlo ** 6 + 32 * rlo ** 7)
        cb = 1 / (3 * rlo ** 3) - w * 3 * rhi ** 3 * rlo ** 6 * (
            7 * rhi ** 4 + 42 * rhi ** 3 * rlo + 112 * rhi ** 2 * rlo ** 2 +
            150 * rhi * rlo ** 3 + 25 * rlo ** 4)
        return 2 * math.pi / V * (ca * A + cb * B)

    def evaluate(self, r, q=None, sig=None, eps=None):
        q = self.q if q is None else q
        sig = self.sig if sig is None else sig
        eps = self.eps if eps is None else eps
        phi, ev, ljf, ulj, w = self.rspace(r, q, sig, eps)
        kphi, kev, ke, kw = self.recip(r, q)
        tail = self.tail(sig, eps)
        phi = phi + kphi - self.p["eta"] * (2 / math.sqrt(math.pi)) * q
        elec = 0.5 * (q * phi).sum()
        f = q[:, None] * (ev + kev) + ljf
        lj = ulj + tail
        vir = w + kw + tail * torch.eye(3, device=self.dev, dtype=torch.float64)
        return f, torch.stack([elec, lj, tail, elec + lj, 0 * elec, ke]), vir

    # -- rigid water and velocity Verlet
    def _gradients(self, x):
        """Constraint values and gradients of waters x [n, 3, 3]."""
        bond, angle = 1.0, math.radians(109.47)
        a, b = x[:, 1] - x[:, 0], x[:, 2] - x[:, 0]
        na, nb = a.norm(dim=1, keepdim=True), b.norm(dim=1, keepdim=True)
        ct = ((a * b).sum(1, keepdim=True) / (na * nb)).clamp(-1, 1)
        st = torch.sqrt(1 - ct * ct)
        g1 = -(b / (na * nb) - a * ct / na ** 2) / st
        g2 = -(a / (na * nb) - b * ct / nb ** 2) / st
        o = torch.zeros_like(a)
        g = torch.stack([torch.stack([-a, a, o], 1), torch.stack([-b, o, b], 1),
                         torch.stack([-g1 - g2, g1, g2], 1)], 1)
        val = torch.cat([0.5 * (na ** 2 - bond ** 2), 0.5 * (nb ** 2 - bond ** 2),
                         torch.acos(ct) - angle], 1)
        return val, g

    def shake(self, x, v, x0, dt):
        im = 1 / self.m[self.g0[self.water][:, None] + torch.arange(3, device=self.dev)]
        _, g0 = self._gradients(x0)
        g0 = g0 * im[:, None, :, None]
        x, v = x.clone(), v.clone()
        for _ in range(50):
            val, g = self._gradients(x)
            todo = torch.nonzero((val.abs() > 1e-8).any(1))[:, 0]
            if not todo.numel():
                break
            S = torch.einsum("naij,nbij->nab", g[todo], g0[todo])
            lam = torch.linalg.solve(S, -val[todo])
            d = (lam[:, :, None, None] * g0[todo]).sum(1)
            x[todo] += d
            if dt:
                v[todo] += d / dt
        return x, v

    def rattle(self, x, v):
        im = 1 / self.m[self.g0[self.water][:, None] + torch.arange(3, device=self.dev)]
        _, g = self._gradients(x)
        gm = g * im[:, None, :, None]
        S = torch.einsum("naij,nbij->nab", g, gm)
        lam = torch.linalg.solve(S, -torch.einsum("naij,nij->na", g, v))
        return v + (lam[:, :, None, None] * gm).sum(1)

    def md(self, r, v, steps):
        at = self.g0[self.water][:, None] + torch.arange(3, device=self.dev)
        r = r.clone()
        r[at] = self.shake(r[at], 0 * r[at], r[at], 0.0)[0]
        self.find_pairs(r, 1.0)
        f, en, _ = self.evaluate(r)
        for k in range(steps):
            v = v + f * (DT / 2 / self.m)[:, None]
            x = r + v * DT
            x[at], vw = self.shake(x[at], v[at], r[at], DT)
            v[at] = vw
            r = x
            if k % 10 == 9:
                self.find_pairs(r, 1.0)
            f, en, _ = self.evaluate(r)
            v = v + f * (DT / 2 / self.m)[:, None]
            v[at] = self.rattle(r[at], v[at])
        en[4] = (0.5 * self.m[:, None] * v * v).sum()
        return r, v, f, en


def _np(x):
    return x.detach().cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "remd":      # draws and exchanges: no closed statement
        return None
    s, p = _system(case, seed)
    mesh = None
    if kind == "dropin" and p["kmode"] == 1:
        n = W.smooth_mesh_size(case["nx"])
        mesh = (n, n, n)
    x = _Exact(case, s, p, mesh)
    t = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device=x.dev)
    r = t(s.r)
    if kind == "md":
        r, v, f, en = x.md(r, t(s.v), case["steps"])
        return dict(r=_np(r), v=_np(v), f=_np(f), energies=_np(en)[None])
    x.find_pairs(r, 0.0)
    if kind == "force":
        f, en, w = x.evaluate(r)
        out = dict(f=_np(f), energies=_np(en)[None])
        if case["virial"]:
            out["virial"] = _np(w)[None]
        return out
    if kind == "grad":
        key = np.stack([s.q, s.sig, s.eps, s.site_mask], 1)
        _, first, inv = np.unique(key, axis=0, return_index=True, return_inverse=True)
        rank = np.argsort(np.argsort(first))
        ty = torch.as_tensor(rank[inv.reshape(-1)], device=x.dev)
        th = t(key[np.sort(first), :3]).requires_grad_(True)
        q, sig, eps = th[ty, 0], th[ty, 1], th[ty, 2]
        f, en, _ = x.evaluate(r, q, sig, eps)
        loss = ((f - t(_f_ref(s, seed))) ** 2).sum()
        dE, = torch.autograd.grad(en[3], th, retain_graph=True)
        dL, = torch.autograd.grad(loss, th)
        lj = np.repeat((key[np.sort(first), 3].astype(int) & 2 != 0)[:, None], 3, 1)
        lj[:, 0] = True
        return dict(dE=np.where(lj, _np(dE), 0.0), dL=np.where(lj, _np(dL), 0.0),
                    loss=float(loss))
    phi, ev, ljf, ulj, _ = x.rspace(r, x.q, x.sig, x.eps)
    kphi, kev, _, _ = x.recip(r, x.q)
    return dict(phi=_np(phi), evec=_np(ev), lj_force=_np(ljf), lj_energy=_np(ulj)[None],
                kphi=_np(kphi), kevec=_np(kev))
