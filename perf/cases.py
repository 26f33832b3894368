"""Performance cases of the H-apply path.

Each case is a piece of work that a program using this package gives it: a Laplacian, a
Hamiltonian apply, a propagation step, a Krylov step, an orthogonalisation or a gradient,
through the entry points of ``octhip.api``, at mesh sizes and state counts of the
workloads, the benchmark and the tests.  ``listed`` holds the fixed cases, ``draw`` more of
the same ranges, ``prepare`` builds the handles and inputs a program holds before the call,
``run`` makes one pass, ``work`` counts the bytes and operations it cannot do without and
``exact`` repeats the pass in plain torch, float64.
"""
from __future__ import annotations

import math
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "octopus-debian-package_amd"))

from octhip import _lib, api, periodic, rng, workloads  # noqa: E402
from octhip.autograd import overlap_objective  # noqa: E402
from octhip.mesh import cube_mesh, sphere_mesh  # noqa: E402
from octhip.projectors import kb_projector_set  # noqa: E402
from octhip.stencil import nl_operator_build, star_points  # noqa: E402


def listed():
    return [
        # the smallest call: a Laplacian of three complex functions on a few thousand
        # points (a small molecule, a test run): launches and latency count
        dict(name="laplacian_small", kind="laplacian", box="sphere", size=3.0, h=0.3, nst=3, cplx=True),
        # the plain finite-difference workload: 64^3 box, 8 real functions
        dict(name="laplacian_cube64", kind="laplacian", box="cube", size=64.0, h=0.3, nst=8, cplx=False),
        # a ground-state H-apply: real wavefunctions, a state count that does not fill its block
        dict(name="happly_real13", kind="happly", size=8.0, h=0.3, nst=13, pack=32, cplx=False, natoms=5),
        # the smallest of the uneven systems: 8 complex states on the R=6 sphere
        dict(name="happly_R6_8", kind="happly", size=6.0, h=0.25, nst=8, pack=32, cplx=True, natoms=16),
        # the headline workload: 64 complex states in blocks of 32 on the R=12 sphere
        dict(name="happly_R12_64", kind="happly", size=12.0, h=0.25, nst=64, pack=32, cplx=True, natoms=16),
        # real-time propagation as one graph per step: 128 states in 4 blocks
        dict(name="taylor_graph_R12_128", kind="graph", size=12.0, h=0.25, nst=128, pack=32, natoms=16, order=4),
        # a driven time step with the density of the propagated states (exponential
        # midpoint), launched eagerly; the second block is half empty
        dict(name="expmid_R10_48", kind="expmid", size=10.0, h=0.3, nst=48, pack=32, natoms=16, order=4),
        # independent systems of uneven size in one launch sequence
        dict(name="batched_uneven4", kind="batched", size=6.0, size2=10.0, systems=4, h=0.25, nst=8, nst2=48,
             natoms=16, order=4),
        # an optimal-control gradient: forward with checkpoints, objective, backward
        dict(name="adjoint_R10_32", kind="adjoint", size=10.0, h=0.3, nst=32, natoms=16, steps=20, every=10),
        # a Lanczos propagation step (Krylov space up to 16)
        dict(name="lanczos_R8_16", kind="lanczos", size=8.0, h=0.25, nst=16, natoms=16, order=16),
        # one k-point of a periodic cell: boundary images and Bloch phases
        dict(name="kpoint_cell40_16", kind="kpoint", size=40.0, h=0.3, nst=16, natoms=4),
        # an eigensolver's inner step: H psi orthogonalised against four blocks, normalised
        dict(name="orthogonalise_R10_32", kind="orthogonalise", size=10.0, h=0.3, nst=32, nvec=4, natoms=16),
    ]


# Radius and state-count ranges of the drawn cases; the state-points of a drawn case stay
# below those of the largest listed case of its kind.
_CAP = dict(laplacian=4e6, happly=30e6, graph=60e6, expmid=7.5e6, batched=8e6, adjoint=5e6, lanczos=4e6, kpoint=1.1e6,
            orthogonalise=5e6)


def draw(r):
    kind = r.choice(["laplacian", "happly", "happly", "happly", "graph", "graph", "expmid", "batched", "adjoint",
                     "lanczos", "kpoint", "orthogonalise"])
    h = r.choice([0.25, 0.3, 0.35, 0.4])
    hi = {"happly": 12.0, "graph": 12.0, "lanczos": 8.0}.get(kind, 10.0)
    size = round(math.exp(r.uniform(math.log(3.0), math.log(hi))), 2)
    nst = int(round(math.exp(r.uniform(0.0, math.log(64.5)))))
    natoms = r.randint(1, 20)
    points = 4.0 / 3.0 * math.pi * (size / h) ** 3
    if kind == "laplacian":
        c = dict(kind=kind, box="sphere", size=size, h=h, nst=nst, cplx=r.random() < 0.5)
        if r.random() < 0.4:
            c.update(box="cube", size=float(r.randint(20, 80)))
            points = c["size"] ** 3
    elif kind == "happly":
        c = dict(kind=kind, size=size, h=h, nst=nst, pack=r.choice([8, 16, 32, 32, 64]), cplx=r.random() < 0.7,
                 natoms=natoms)
    elif kind in ("graph", "expmid"):
        c = dict(kind=kind, size=size, h=h, nst=nst, pack=r.choice([16, 32, 32]), natoms=natoms,
                 order=r.choice([4, 4, 4, 2, 6]))
    elif kind == "batched":
        size2 = round(min(size * r.uniform(1.2, 2.0), 10.0), 2)
        c = dict(kind=kind, size=size, size2=size2, systems=r.randint(2, 5), h=h, nst=r.randint(1, 16),
                 nst2=r.randint(8, 48), natoms=natoms, order=r.choice([4, 4, 2]))
        nst, points = c["nst2"], c["systems"] * 4.0 / 3.0 * math.pi * (size2 / h) ** 3 / 2.0
    elif kind == "adjoint":
        c = dict(kind=kind, size=size, h=h, nst=min(nst, 32), natoms=natoms, steps=r.randint(3, 20), every=r.randint(2, 10))
        nst = c["nst"]
    elif kind == "lanczos":
        c = dict(kind=kind, size=size, h=h, nst=min(nst, 32), natoms=natoms, order=r.randint(14, 20))
        nst = c["nst"]
    elif kind == "kpoint":
        c = dict(kind=kind, size=float(r.randint(20, 48)), h=h, nst=min(nst, 32), natoms=r.randint(1, 6))
        nst, points = c["nst"], c["size"] ** 3
    else:
        c = dict(kind=kind, size=size, h=h, nst=min(nst, 32), nvec=r.randint(1, 6), natoms=natoms)
        nst, points = c["nst"], points * max(1.0, c["nvec"] / 4.0)
    # too many state-points: fewer states
    if points * nst > _CAP[kind]:
        key = "nst2" if kind == "batched" else "nst"
        c[key] = max(1, int(_CAP[kind] / points))
    return c


# ------------------------------------------------------------------- inputs --
# Meshes and stencil tables depend on the geometry alone: a program builds them once.
_meshes = {}


def _mesh(box, size, h):
    key = (box, size, h)
    if key not in _meshes:
        while len(_meshes) >= 12:
            del _meshes[next(iter(_meshes))]
        if box == "sphere":
            m = sphere_mesh(size, h, star_points(4))
        else:
            m = cube_mesh(int(size), h, star_points(4))
        _meshes[key] = (m, nl_operator_build(m, 4))
    return _meshes[key]


def _system(size, h, natoms, seed):
    """Gaussian wells and KB atoms (l <= 1) at seeded sites inside a sphere."""
    mesh, op = _mesh("sphere", size, h)
    rc = min(3.0, 0.4 * size)
    inner = size - rc
    v = workloads.gaussian_wells(mesh, rng.in_ball(seed, 1, 16, inner))
    alphas = rng.uniform(seed, 3, natoms * 2, 0.6, 1.2).reshape(natoms, 2)
    energies = rng.uniform(seed, 4, natoms * 2, -1.0, 1.0).reshape(natoms, 2)
    proj = kb_projector_set(mesh, rng.in_ball(seed, 2, natoms, inner), rc, alphas, energies)
    return workloads.System(mesh=mesh, op=op, v=v, proj=proj, seed=seed, name="case")


def _cell(size, h, natoms, seed):
    n = int(size)
    return periodic.periodic_system(n=n, spacing=h, natoms=natoms, nwells=4, rc=0.18 * n * h, seed=seed)


def _blocks(nst, pack):
    """(states, block size) of each packed batch: full blocks, then the remainder."""
    if nst <= pack:
        return [(nst, api.pad_pow2(nst))]
    return [(min(pack, nst - f), pack) for f in range(0, nst, pack)]


def _states(mesh, nst, pack, cplx, seed, scale=3.0):
    """A packed block (np_part rows) of seeded states under a Gaussian envelope; padding
    states and boundary rows are zero."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.from_numpy(mesh.x[: mesh.np]).cuda()
    r2 = (x * x).sum(1)
    env = torch.exp(-r2 / (r2.max() / scale))
    k = 2 if cplx else 1
    ff = torch.zeros((mesh.np_part, k * pack), dtype=torch.float64, device="cuda")
    ff[: mesh.np, : k * nst] = torch.randn((mesh.np, k * nst), generator=g, dtype=torch.float64, device="cuda") * env[:, None]
    return ff


def _batch(mesh, nst, pack, cplx, seed, normalise=False):
    ff = _states(mesh, nst, pack, cplx, seed)
    if normalise:
        z = torch.view_as_complex(ff[:, : 2 * nst].reshape(-1, nst, 2).contiguous())
        z = z / torch.sqrt(mesh.vol_pp * (z.abs() ** 2).sum(0))
        ff[:, : 2 * nst] = torch.view_as_real(z).reshape(-1, 2 * nst)
    return api.Batch(nst, mesh.np_part, cplx, pack, ff=ff)


def _uneven(case):
    """(radius, states) of each system of a batched case, growing geometrically."""
    n = case["systems"]
    t = [i / max(n - 1, 1) for i in range(n)]
    return [(round(case["size"] * (case["size2"] / case["size"]) ** u, 2),
             max(1, int(round(case["nst"] * (max(case["nst2"], 1) / case["nst"]) ** u)))) for u in t]


def _dt(case):
    return 0.2 * case["h"] ** 2  # inside Taylor-4's stability bound of the order-4 star


K_POINT = (0.3, -0.2, 0.45)
FIELD = (0.004, -0.002, 0.003)


def _inputs(case, seed):
    """Everything seeded of a case, without handles: systems, state blocks, weights."""
    kind = case["kind"]
    s = SimpleNamespace(kind=kind, case=case)
    if kind == "laplacian":
        s.mesh, s.op = _mesh(case["box"], case["size"], case["h"])
        s.parts = [(case["nst"], api.pad_pow2(case["nst"]))]
        s.batches = [_batch(s.mesh, n, p, case["cplx"], seed) for n, p in s.parts]
        return s
    if kind == "batched":
        s.systems = []
        for i, (radius, nst) in enumerate(_uneven(case)):
            sy = _system(radius, case["h"], case["natoms"], seed * 16 + i)
            s.systems.append((sy, [_batch(sy.mesh, n, p, True, seed * 64 + 8 * i + j, True)
                                   for j, (n, p) in enumerate(_blocks(nst, 32))]))
        return s
    s.system = _cell(case["size"], case["h"], case["natoms"], seed) if kind == "kpoint" else _system(
        case["size"], case["h"], case["natoms"], seed)
    s.mesh = s.system.mesh
    cplx = case.get("cplx", True)
    s.parts = _blocks(case["nst"], case.get("pack", 32))
    s.batches = [_batch(s.mesh, n, p, cplx, seed * 64 + j, kind not in ("happly", "kpoint"))
                 for j, (n, p) in enumerate(s.parts)]
    if kind == "expmid":
        s.weights = [list(rng.uniform(seed, 20 + j, n, 0.5, 2.0)) for j, (n, p) in enumerate(s.parts)]
    if kind == "adjoint":
        n, p = s.parts[0]
        s.target = _batch(s.mesh, n, p, True, seed * 64 + 50, True)
        w, a, ph = workloads.dipole_field(seed)
        s.eps = workloads.eps_of_t((np.arange(case["steps"]) + 0.5) * _dt(case), w, a, ph)
    if kind == "orthogonalise":
        n, p = s.parts[0]
        s.vecs = [_batch(s.mesh, n, p, True, seed * 64 + 30 + k, True) for k in range(case["nvec"])]
    return s


def prepare(case, seed):
    _lib.init(0)
    s = _inputs(case, seed)
    kind = s.kind
    if kind == "laplacian":
        s.dev = api.NLOperatorDevice(s.op, star_points(4))
        s.out = [api.Batch(n, s.mesh.np, case["cplx"], p) for n, p in s.parts]
        return s
    if kind == "batched":
        s.hms = [api.HamiltonianDevice.from_system(sy) for sy, _ in s.systems]
        pairs = [(hm, b) for hm, (_, bs) in zip(s.hms, s.systems) for b in bs]
        s.prop = api.BatchedPropagator(pairs, _dt(case), order=case["order"], with_apply=False)
        s.results = [b.ff for _, b in pairs]
        return s
    if kind == "kpoint":
        s.hm = api.HamiltonianDevice(api.NLOperatorDevice(s.system.op, star_points(4)), s.system.v, s.system.proj)
        s.hm.set_periodic(s.system.bnd_src)
        phase, corr = s.system.phases(K_POINT)
        s.hm.set_phases(phase, corr, s.system.pphase_of(K_POINT))
    else:
        s.hm = api.HamiltonianDevice.from_system(s.system)
    if kind in ("happly", "kpoint", "orthogonalise"):
        s.out = [api.Batch(n, s.mesh.np, case.get("cplx", True), p) for n, p in s.parts]
    elif kind == "graph":
        s.te = api.Exponential(case["order"])
        s.graph = api.TaylorGraph(s.te, s.hm, s.batches, _dt(case))
    elif kind == "expmid":
        s.te = api.Exponential(case["order"])
        s.hm.set_dipole_field((0.0, 0.0, 0.0), s.mesh.x[: s.mesh.np])
        s.density = torch.zeros(s.mesh.np, dtype=torch.float64, device="cuda")
    elif kind == "adjoint":
        s.adj = api.Adjoint(s.hm, s.mesh.x, (1.0, 0.0, 0.0), s.batches[0].ldf, case["steps"], _dt(case), s.mesh.vol_pp,
                            checkpoint_every=case["every"])
    elif kind == "lanczos":
        s.te = api.Exponential(case["order"], method="lanczos")
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s.kind
    if kind == "laplacian":
        for fi, fo in zip(s.batches, s.out):
            api.nl_operator_operate_batch(s.dev, fi, fo)
        return [b.ff for b in s.out]
    if kind in ("happly", "kpoint"):
        for b, o in zip(s.batches, s.out):
            api.hamiltonian_elec_apply_batch(s.hm, b, o)
        return [b.ff for b in s.out]
    if kind == "graph":
        s.graph.launch()
        return [b.ff[: s.mesh.np] for b in s.batches]
    if kind == "expmid":
        api.propagator_expmid(s.te, s.hm, s.batches, _dt(s.case), FIELD, s.weights, s.density)
        return [b.ff[: s.mesh.np] for b in s.batches] + [s.density]
    if kind == "batched":
        s.prop.taylor_step()
        return [f[: hm.np] for f, (hm, _) in zip(s.results, s.prop.pairs)]
    if kind == "adjoint":
        psi = s.batches[0].clone()
        s.adj.forward(psi, s.eps)
        J, chi = overlap_objective(s.target, psi, s.mesh.np, s.mesh.vol_pp)
        deps, dv = s.adj.backward(chi)
        return [psi.ff[: s.mesh.np], J, chi.ff[: s.mesh.np], deps, dv]
    if kind == "lanczos":
        for b in s.batches:
            s.te.apply_batch(s.hm, b, 2.5 * _dt(s.case))
        return [b.ff[: s.mesh.np] for b in s.batches]
    api.hamiltonian_elec_apply_batch(s.hm, s.batches[0], s.out[0])
    overlap, norm = api.mesh_batch_orthogonalization(s.mesh.vol_pp, s.vecs, s.out[0], s.mesh.np, normalize=True)
    return [s.out[0].ff, overlap, norm]


# --------------------------------------------------------------------- work --
def work(case):
    """Compulsory bytes and operations: every state row read and written once per H-apply
    (which the next one cannot start without), the potential and the projectors once."""
    kind = case["kind"]

    def happly(mesh, nst, es, natoms, rc):
        pts = natoms * 4.0 / 3.0 * math.pi * (rc / mesh.spacing) ** 3
        lanes = nst * es / 8
        return (es * nst * (mesh.np_part + mesh.np) + 8 * mesh.np + pts * (8 * 4 + 12),
                lanes * (mesh.np * 52 + pts * 16))

    if kind == "laplacian":
        mesh, _ = _mesh(case["box"], case["size"], case["h"])
        es = 16 if case["cplx"] else 8
        return {"bytes": es * case["nst"] * (mesh.np_part + mesh.np) + 200, "flops": 50 * mesh.np * case["nst"] * es / 8}
    if kind == "kpoint":
        n = int(case["size"])
        mesh = SimpleNamespace(np=n ** 3, np_part=n ** 3 + 24 * n * n, spacing=case["h"])
        b, f = happly(mesh, case["nst"], 16, case["natoms"], 0.18 * n * case["h"])
        return {"bytes": b + 16 * mesh.np_part, "flops": f + 12 * mesh.np_part * case["nst"]}
    if kind == "batched":
        b = f = 0.0
        for radius, nst in _uneven(case):
            mesh, _ = _mesh("sphere", radius, case["h"])
            x, y = happly(mesh, nst, 16, case["natoms"], min(3.0, 0.4 * radius))
            b, f = b + case["order"] * x, f + case["order"] * y
        return {"bytes": b, "flops": f}
    mesh, _ = _mesh("sphere", case["size"], case["h"])
    nst = case["nst"]
    es = 16 if case.get("cplx", True) else 8
    b, f = happly(mesh, nst, es, case["natoms"], min(3.0, 0.4 * case["size"]))
    rows = es * nst * mesh.np
    if kind == "happly":
        return {"bytes": b, "flops": f}
    if kind in ("graph", "expmid"):
        return {"bytes": case["order"] * b, "flops": case["order"] * (f + 8 * mesh.np * nst)}
    if kind == "adjoint":
        # forward and backward propagation, and the contraction of the two
        return {"bytes": case["steps"] * (8 * b + 2 * rows), "flops": case["steps"] * (8 * f + 80 * mesh.np * nst)}
    if kind == "lanczos":
        # about ten Krylov steps: an H-apply, the overlaps with two vectors and the update
        return {"bytes": 10 * (b + 3 * rows), "flops": 10 * (f + 24 * mesh.np * nst)}
    return {"bytes": b + case["nvec"] * rows, "flops": f + 16 * case["nvec"] * mesh.np * nst}


# -------------------------------------------------------------------- exact --
_C8 = [-205.0 / 72.0, 8.0 / 5.0, -1.0 / 5.0, 8.0 / 315.0, -1.0 / 560.0]  # 8th-order second derivative


class _H:
    """-1/2 Laplacian + v + KB projectors in plain torch (float64 rows of lanes)."""

    def __init__(self, mesh, v=None, proj=None, factor=-0.5, bnd=None, pphase=None):
        self.mesh, self.factor = mesh, factor
        c = torch.from_numpy(mesh.coords.astype(np.int64)).cuda()
        lo, hi = c.min(0).values - 4, c.max(0).values + 4
        n = hi - lo + 1
        site = lambda q: ((q[:, 0] - lo[0]) * n[1] + (q[:, 1] - lo[1])) * n[2] + (q[:, 2] - lo[2])  # noqa: E731
        table = torch.full((int(n.prod()),), -1, dtype=torch.int64, device="cuda")
        table[site(c)] = torch.arange(mesh.np_part, device="cuda")
        ci = c[: mesh.np]
        self.terms = [(3.0 * _C8[0], None)]
        for d in range(3):
            for k in (-4, -3, -2, -1, 1, 2, 3, 4):
                off = torch.zeros(3, dtype=torch.int64, device="cuda")
                off[d] = k
                self.terms.append((_C8[abs(k)], table[site(ci + off)]))
        self.v = None if v is None else torch.from_numpy(np.asarray(v)).cuda()
        self.bnd = None if bnd is None else torch.from_numpy(bnd.astype(np.int64)).cuda()
        self.mats = []
        for a in range(0 if proj is None else proj.nmat):
            P, m, sc = proj.matrix(a)
            o = int(proj.offsets[a][3])
            ph = None if pphase is None else torch.from_numpy(pphase[o:o + len(m)]).cuda()
            self.mats.append((torch.from_numpy(np.ascontiguousarray(P)).cuda(),
                              torch.from_numpy(m.astype(np.int64) - 1).cuda(), torch.from_numpy(np.array(sc)).cuda(), ph))

    def full(self, x):
        """np rows -> np_part rows: zero boundary, or the periodic images."""
        nb = self.mesh.np_part - self.mesh.np
        if self.bnd is not None:
            return torch.cat([x, x[self.bnd]])
        return torch.cat([x, torch.zeros((nb, x.shape[1]), dtype=x.dtype, device="cuda")])

    def __call__(self, x, rows=None):
        f = self.full(x) if rows is None else rows
        h2 = self.factor / self.mesh.spacing ** 2
        out = (h2 * self.terms[0][0]) * f[: self.mesh.np]
        for w, idx in self.terms[1:]:
            out = out + (h2 * w) * f[idx]
        if self.v is not None:
            out = out + self.v[:, None] * f[: self.mesh.np]
        cx = f.is_complex()
        for P, m, sc, ph in self.mats:
            g = f[m] if ph is None else ph[:, None] * f[m]
            g = torch.view_as_real(g).reshape(len(m), -1) if cx else g
            k = P @ (sc[:, None] * (P.t().contiguous() @ g))
            k = torch.view_as_complex(k.reshape(len(m), -1, 2).contiguous()) if cx else k
            out[m] += k if ph is None else torch.conj(ph)[:, None] * k
        return out


def _rows(batch, rows):
    return torch.view_as_complex(batch.ff[:rows].reshape(rows, batch.pack_size, 2).contiguous()) if batch.is_complex else batch.ff[:rows]


def _flat(z):
    return torch.view_as_real(z).reshape(z.shape[0], -1) if z.is_complex() else z


def _taylor(h, z, dt, order, powers=None):
    y, c, out = z, 1.0 + 0.0j, z
    for k in range(1, order + 1):
        if powers is not None:
            powers.append(y)
        y = h(y)
        c = c * (-1j * dt) / k
        out = out + c * y
    return out


def exact(case, seed):
    s = _inputs(case, seed)
    kind = s.kind
    if kind == "laplacian":
        h = _H(s.mesh, factor=1.0)
        return [_flat(h(_rows(b, s.mesh.np))) for b in s.batches]
    if kind == "batched":
        out = []
        for sy, bs in s.systems:
            h = _H(sy.mesh, sy.v, sy.proj)
            out += [_flat(_taylor(h, _rows(b, sy.mesh.np), _dt(case), case["order"])) for b in bs]
        return out
    n, mesh = s.mesh.np, s.mesh
    if kind == "kpoint":
        ph, _ = s.system.phases(K_POINT)
        ph = torch.from_numpy(ph).cuda()[:, None]
        h = _H(mesh, s.system.v, s.system.proj, bnd=s.system.bnd_src, pphase=s.system.pphase_of(K_POINT))
        return [_flat(torch.conj(ph[:n]) * h(None, rows=ph * h.full(_rows(b, n)))) for b in s.batches]
    h = _H(mesh, s.system.v, s.system.proj)
    if kind == "happly":
        return [_flat(h(_rows(b, n))) for b in s.batches]
    if kind == "graph":
        return [_flat(_taylor(h, _rows(b, n), _dt(case), case["order"])) for b in s.batches]
    x = torch.from_numpy(mesh.x[:n]).cuda()
    v0 = h.v
    if kind == "expmid":
        h.v = v0 + x @ torch.tensor(FIELD, dtype=torch.float64, device="cuda")
        out = [_taylor(h, _rows(b, n), _dt(case), case["order"]) for b in s.batches]
        rho = sum((z[:, : len(w)].abs() ** 2 @ torch.tensor(w, dtype=torch.float64, device="cuda")) for z, w in zip(out, s.weights))
        return [_flat(z) for z in out] + [rho]
    if kind == "adjoint":
        dt, vol, order = _dt(case), mesh.vol_pp, 4
        psi, kept = _rows(s.batches[0], n), []
        for e in s.eps:
            h.v = v0 + e * x[:, 0]
            kept.append([])
            psi = _taylor(h, psi, dt, order, kept[-1])
        phi = _rows(s.target, n)
        ov = vol * (torch.conj(phi) * psi).sum(0)
        chi = phi * ov[None, :]
        dv = torch.zeros(n, dtype=torch.float64, device="cuda")
        deps = np.zeros(len(s.eps))
        zf = [(-1j * dt) ** k / math.factorial(k) for k in range(order + 1)]
        for t in reversed(range(len(s.eps))):
            h.v = v0 + s.eps[t] * x[:, 0]
            back = []
            nxt = _taylor(h, chi, -dt, order, back)
            rho = torch.zeros(n, dtype=torch.float64, device="cuda")
            for m in range(order):
                u = sum(zf[m + k + 1] * kept[t][k] for k in range(order - m))
                rho += (torch.conj(back[m]) * u).real.sum(1)
            dv += 2.0 * vol * rho
            deps[t] = 2.0 * vol * float((x[:, 0] * rho).sum())
            chi = nxt
        # the gradients' chi_0 replaces chi_N in the batch
        return [_flat(psi), (ov.abs() ** 2).sum(), _flat(chi), deps, dv]
    if kind == "lanczos":
        return [_flat(_taylor(h, _rows(b, n), 2.5 * _dt(case), 40)) for b in s.batches]
    z = h(_rows(s.batches[0], n))
    nst = s.batches[0].nst
    vecs = [_rows(b, n) for b in s.vecs]
    ov = [mesh.vol_pp * (torch.conj(q) * z).sum(0) for q in vecs]
    for q, o in zip(vecs, ov):
        z = z - q * o[None, :]
    norm = torch.sqrt(mesh.vol_pp * (z.abs() ** 2).sum(0))[:nst]
    z[:, :nst] = z[:, :nst] / norm[None, :]
    return [_flat(z), torch.stack([o[:nst] for o in ov]).cpu().numpy(), norm.cpu().numpy()]
