"""Performance cases of the EBE-PCG + viscoplastic path on one GPU.

Every case is work that a user of the package has it do, through its public
entry points, on slopes of the repository's own benchmark family (two layers
split at z = 10 m, jittered interior nodes, base fixed, side rollers), from
the 1,152-element mesh up to the 144,000-element one, with odd and ragged
grids among them:

* ``dropin``    pcg_solver, the reference's solver seam: host arrays in the
                reference layout, the element matrices cached on the device;
* ``solve``     DeviceMesh.solve on the resident mesh, full or packed FP64;
* ``plastic``   a strength-reduction trial's plastic iterations, from the
                reset to the result fields (DeviceSlope);
* ``batch``     one plastic iteration of many trials at once on the
                mixed-precision engine (BatchEngine), 1 to 64 columns;
* ``analyses``  whole factor-of-safety sweeps on the engine (run_analyses);
* ``setup``     a request's set-up: numbering, resident mesh, stiffness;
* ``stage``     what an excavation stage computes from the stress state.

Solves run either to a tight tolerance, so that the result is the system's
solution and not the place where the stop test fell, or for a fixed count of
iterations (``cap``) where a full solve would take seconds.  Materials,
strengths, jitter and so the right-hand sides come from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from specfem3d_geotech_amd.batch import (DEFAULT_INNER_TOL, Analysis, BatchEngine,
                                         device_mesh, run_analyses)
from specfem3d_geotech_amd.mesh import Material, slope_mesh
from specfem3d_geotech_amd.plastic import dt_viscoplas, strength_reduction
from specfem3d_geotech_amd.slope import DeviceSlope
from specfem3d_geotech_amd.solver import (K_F64, KFMT_FULL, KFMT_PACKED, Context,
                                          DeviceMesh, pcg_solver)
from specfem3d_geotech_amd.spec import hex2spec_device

NL_TOL = 5e-4       # the tolerance of every configuration
MAXITER = 20000
TIGHT = 2e-13


def listed():
    return [
        # The drop-in on the small benchmark mesh (24x4x12, 1,152 elements):
        # launch latency sets the time of an iteration.
        dict(name="dropin_1k", kind="dropin", nx=24, ny=4, nz=12, tol=1e-11, cap=0),
        # Resident FP64 solves: a ragged mid-size mesh on the packed operator,
        # the large full-storage operator, and the 144,000-element mesh packed.
        dict(name="solve_packed_5k", kind="solve", nx=37, ny=7, nz=19, packed=True,
             tol=1e-11, cap=0),
        dict(name="solve_full_30k", kind="solve", nx=66, ny=13, nz=35, packed=False,
             tol=1e-10, cap=200),
        dict(name="solve_packed_144k", kind="solve", nx=120, ny=20, nz=60, packed=True,
             tol=1e-10, cap=120),
        # One trial's plastic iterations on the packed FP64 operator, with the
        # state and result fields that a sweep saves at the end of an SRF.
        dict(name="plastic_9k", kind="plastic", nx=45, ny=9, nz=23, packed=True, srf=1.25),
        # The mixed engine: one column (an excavation increment's form) on a
        # mid-size mesh, 8 columns (a served request), 64 columns (strength
        # realisations) on a large and on the small benchmark mesh.
        dict(name="batch1_6k", kind="batch", nx=30, ny=10, nz=21, ncol=1, srf=1.2),
        dict(name="batch8_25k", kind="batch", nx=64, ny=12, nz=33, ncol=8, srf=1.2),
        dict(name="batch64_12k", kind="batch", nx=56, ny=8, nz=28, ncol=64, srf=1.2),
        dict(name="batch64_1k", kind="batch", nx=24, ny=4, nz=12, ncol=64, srf=1.2),
        # Whole sweeps of 8 realisations on a small mesh, as the scheduler
        # runs them.
        dict(name="analyses_400", kind="analyses", nx=16, ny=3, nz=8, ncol=8, count=8),
        # A request's set-up, and an excavation stage's element kernels.
        dict(name="setup_63k", kind="setup", nx=90, ny=15, nz=47),
        dict(name="stage_19k", kind="stage", nx=57, ny=11, nz=31),
    ]


def draw(rng):
    """A case of the same ranges: grids of 300 to 60,000 elements (to 16,000
    where 64 columns run), aspect ratios around the benchmark's 6:1:3."""
    kind = rng.choice(["dropin", "solve", "solve", "plastic", "batch", "batch", "batch",
                       "analyses", "setup", "stage"])
    ncol = rng.choice([1, 2, 4, 8, 16, 32, 64])
    top = {"dropin": 6000, "solve": 60000, "plastic": 9000, "analyses": 700,
           "setup": 60000, "stage": 19000,
           "batch": 24000 if ncol <= 8 else 12000}[kind]
    ne = math.exp(rng.uniform(math.log(300), math.log(top)))
    nx = max(6, int(round((2.0 * 6.0 * ne) ** (1 / 3) * rng.uniform(0.9, 1.15))))
    ny = max(2, int(round(nx / rng.uniform(4.0, 7.0))))
    nz = max(3, int(round(ne / (nx * ny))))
    while nx * ny * nz > top:
        nz -= 1
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz)
    if kind in ("dropin", "solve"):
        case.update(tol=1e-11, cap=0 if kind == "dropin" or ne < 6000 else rng.randint(60, 200))
    if kind in ("solve", "plastic"):
        case["packed"] = rng.random() < 0.6
    if kind in ("plastic", "batch"):
        case["srf"] = round(rng.uniform(1.0, 1.4), 2)
    if kind == "batch":
        case["ncol"] = ncol
    if kind == "analyses":
        case.update(ncol=8, count=rng.randint(3, 8))
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _mesh(case, seed):
    """The slope with this seed's jitter and moduli."""
    rng = np.random.default_rng(seed)
    mats = [Material(gam=float(rng.uniform(18, 21)), ym=float(rng.uniform(0.8e5, 1.3e5)),
                     nu=float(rng.uniform(0.25, 0.33)), phi=phi * float(rng.uniform(0.95, 1.05)),
                     coh=coh * float(rng.uniform(0.95, 1.05)), psi=0.0)
            for phi, coh in ((25.0, 8.0), (30.0, 20.0))]
    return slope_mesh(case["nx"], case["ny"], case["nz"], materials=mats, layer_z=[10.0],
                      jitter=0.02, seed=seed)


def _strengths(case, mesh, seed):
    """Each trial's factored strengths: lognormal c and tan(phi) around the
    layers' values (coefficients of variation 0.15 and 0.1)."""
    rng = np.random.default_rng([seed, 7])
    _, ym, nu, phi, coh, psi = mesh.material_arrays()
    out = []
    for _ in range(case.get("ncol", 1) if case["kind"] == "batch" else case.get("count", 1)):
        c = coh * math.exp(0.15 * rng.standard_normal())
        t = np.degrees(np.arctan(np.tan(np.radians(phi)) * math.exp(0.1 * rng.standard_normal())))
        out.append((c, t, psi.copy()))
    return out


def _factored(case, mesh, strengths, srf):
    _, ym, nu, *_ = mesh.material_arrays()
    coh, phi, psi = strengths
    cohf, nuf, phif, psif, _ = strength_reduction(srf, False, coh, nu, phi, psi)
    return dict(ym=ym, nuf=nuf, phif=phif, cohf=cohf, psif=psif,
                dt=dt_viscoplas(nuf, phif, ym))


def _stress0(case, mesh, seed):
    """A stress state (nelmt, 27, 6) as an excavation carries it: the
    overburden at each element's depth, perturbed point by point."""
    rng = np.random.default_rng([seed, 11])
    z = mesh.coord[mesh.conn - 1, 2].mean(axis=1)
    szz = -20.0 * (20.0 - z)
    st = np.zeros((mesh.nelmt, 27, 6))
    st[:, :, :3] = (szz[:, None] * np.array([0.5, 0.5, 1.0]))[:, None, :]
    return st + rng.normal(0.0, 2.0, st.shape)


_ctx = None


def _context():
    global _ctx
    if _ctx is None:
        _ctx = Context(0)
    return _ctx


def prepare(case, seed):
    kind = case["kind"]
    ctx = _context()
    mesh = _mesh(case, seed)
    s = dict(case=case, ctx=ctx, mesh=mesh)
    if kind == "setup":
        return s
    if kind == "stage":
        spec = hex2spec_device(ctx, mesh)
        s.update(dm=DeviceMesh(ctx, spec, 2), stress=_stress0(case, mesh, seed),
                 x=np.random.default_rng([seed, 5]).normal(0, 1e-2, spec.neq + 1))
        s["x"][0] = 0.0
        return s
    dm, ext = device_mesh(ctx, mesh)
    s.update(dm=dm, ext=ext)
    if kind == "dropin":
        sp = dm.spec
        gam, ym, nu, *_ = mesh.material_arrays()
        _, dinv = dm.build_stiffness(gam, ym, nu)
        s.update(k=dm.download_stiffness(), dinv=dinv, u0=np.zeros(sp.neq + 1),
                 gdof=np.ascontiguousarray(sp.gdof_elmt, np.int32), neq=sp.neq, nelmt=sp.nelmt)
        dm.close()
        return s
    if kind == "batch" or kind == "analyses":
        s["eng"] = BatchEngine(dm, ext, case["ncol"])
        s["strengths"] = _strengths(case, mesh, seed)
    if kind == "batch":
        s["trials"] = [_factored(case, mesh, t, case["srf"]) for t in s["strengths"]]
        # the elastic solution that every trial of the mesh starts from is
        # solved once per engine
        one = s["eng"]
        one.begin(0, **s["trials"][0])
        one.plastic_iter(np.zeros(case["ncol"], np.int32), TIGHT, MAXITER, DEFAULT_INNER_TOL,
                         NL_TOL)
        one.release(0)
    else:
        dm.set_operator(K_F64, KFMT_PACKED if case.get("packed") else KFMT_FULL)
    if kind == "plastic":
        s["trial"] = _factored(case, mesh, _strengths(case, mesh, seed)[0], case["srf"])
        s["st"] = DeviceSlope(dm, ext)
        dm.ensure_nodes()
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "dropin":
        u, *_ = pcg_solver(s["ctx"], s["neq"], s["nelmt"], s["k"], s["u0"], s["ext"], s["dinv"],
                           s["gdof"], case["tol"], case["cap"] or MAXITER)
        return {"u": u}
    if kind == "solve":
        u, *_ = s["dm"].solve(s["ext"], cg_tol=case["tol"], cg_maxiter=case["cap"] or MAXITER)
        return {"u": u}
    if kind == "plastic":
        st = s["st"]
        st.begin_srf(**s["trial"])
        st.plastic_iter(TIGHT, MAXITER, NL_TOL, False)
        r = st.plastic_iter(TIGHT, MAXITER, NL_TOL, True)
        out = st.download()
        f = st.nodal_fields()
        return dict(out, fmax=r["fmax"], sig=f["stress"], psigma=f["psigma"],
                    nsigma=f["nsigma"])
    if kind == "batch":
        eng, n = s["eng"], case["ncol"]
        for j, t in enumerate(s["trials"]):
            eng.begin(j, **t)
        # the first plastic iteration starts from the engine's elastic
        # solution; the second is every trial's own solve
        eng.plastic_iter(np.zeros(n, np.int32), TIGHT, MAXITER, DEFAULT_INNER_TOL, NL_TOL)
        r = eng.plastic_iter(np.ones(n, np.int32), TIGHT, MAXITER, DEFAULT_INNER_TOL, NL_TOL)
        got = [eng.download(j) for j in range(n)]
        for j in range(n):
            eng.release(j)
        return {"x": np.stack([g[0] for g in got]), "flags": np.stack([g[1] for g in got]),
                "fmax": r["fmax"]}
    if kind == "analyses":
        mesh = s["mesh"]
        _, ym, nu, *_ = mesh.material_arrays()
        an = [Analysis(coh=c, phi=p, psi=q, srf=[0.8, 0.9], tag=i)
              for i, (c, p, q) in enumerate(s["strengths"])]
        run_analyses(s["eng"], an, ym=ym, nu=nu, cg_tol=TIGHT, cg_maxiter=MAXITER,
                     nl_tol=NL_TOL, nl_maxiter=12, keep_state=True)
        return {"x": np.stack([a.x_last for a in an])}
    if kind == "setup":
        mesh, ctx = s["mesh"], s["ctx"]
        spec = hex2spec_device(ctx, mesh)
        gam, ym, nu, *_ = mesh.material_arrays()
        dm = DeviceMesh(ctx, spec, len(gam))
        ext, dinv = dm.build_stiffness(gam, ym, nu)
        dm.close()
        return {"extload": ext, "dinv": dinv, "gdof_elmt": spec.gdof_elmt,
                "g_coord": spec.g_coord}
    _, ym, nu, *_ = s["mesh"].material_arrays()
    gam = s["mesh"].material_arrays()[0]
    st = s["dm"].elastic_stress(ym, nu, s["x"])
    load = s["dm"].excavation_load(gam, s["stress"])
    return {"stress": st, "load": load}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _iterations(case, tol):
    # CG iterations of these slopes: about 12 per element along x at 1e-8
    return 12 * case["nx"] * math.log10(tol) / -8


def work(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    e = nx * ny * nz
    n = 3 * (2 * nx + 1) * (2 * ny + 1) * 2 * nz
    kind = case["kind"]
    # an element's operator from its corners: gather and scatter through its
    # 81 equation numbers, about 5,500 operations per column
    geom, ops = e * (24 * 8 + 81 * 4), 5500.0 * e
    if kind in ("dropin", "solve"):
        its = case["cap"] or _iterations(case, case["tol"])
        # p, r and u read and written once per iteration; the matrices where
        # the caller's own (or the reference-layout) matrices are the operator
        full = kind == "dropin" or not case["packed"]
        per = e * 6561 * 8 + e * 81 * 4 if full else geom
        fl = 2.0 * 6561 * e if full else ops
        return {"bytes": its * (per + 6 * 8 * n) + 24 * n, "flops": its * (fl + 12.0 * n)}
    if kind == "plastic":
        its = 2 * _iterations(case, TIGHT)
        return {"bytes": its * (geom + 6 * 8 * n) + 4 * e * 27 * 48 + 100 * n,
                "flops": its * (ops + 12.0 * n) + 2 * e * 27 * 600.0}
    if kind == "batch":
        b, its = case["ncol"], _iterations(case, TIGHT)
        # r and p in FP32 read and written once, x every eighth iteration
        return {"bytes": its * (geom + b * n * (4 * 4 + 16 / 8)) + b * (4 * e * 27 * 48 + 40 * n),
                "flops": its * b * (ops + 10.0 * n)}
    if kind == "analyses":
        b, its = case["count"], 20 * _iterations(case, TIGHT)
        return {"bytes": its * (geom + b * n * 18), "flops": its * b * (ops + 10.0 * n)}
    if kind == "setup":
        return {"bytes": e * (6561 * 8 + 24 * 8 + 81 * 8 + 27 * 4) + 16 * n,
                "flops": 27.0 * 6561 * 7 * e}
    return {"bytes": e * (2 * 27 * 48 + 24 * 8 + 81 * 4) + 16 * n, "flops": 2 * 27 * 600.0 * e}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
_G = np.array([-1.0, 0.0, 1.0])
_W = np.array([1.0, 4.0, 1.0]) / 3.0
_D = np.array([[-1.5, 2.0, -0.5], [-0.5, 0.0, 0.5], [0.5, -2.0, 1.5]])
_CORNER = np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1],
                    [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]], float)


class _Plain:
    """The discretisation of a structured slope grid: 27-node elements,
    equations numbered by first appearance, element matrices."""

    def __init__(self, case, seed):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        self.places = None
        self.mesh = mesh = _mesh(case, seed)
        self.dev = dev = "cuda" if torch.cuda.is_available() else "cpu"
        ek, ej, ei = (a.ravel() for a in np.meshgrid(np.arange(nz), np.arange(ny),
                                                     np.arange(nx), indexing="ij"))
        lk, lj, li = (a.ravel() for a in np.meshgrid(*[np.arange(3)] * 3, indexing="ij"))
        I, J, K = (2 * a[:, None] + b[None, :] for a, b in ((ei, li), (ej, lj), (ek, lk)))
        gid = I + (2 * nx + 1) * (J + (2 * ny + 1) * K)
        _, first, inv = np.unique(gid.ravel(), return_index=True, return_inverse=True)
        rank = np.empty(first.size, np.int64)
        rank[np.argsort(first, kind="stable")] = np.arange(first.size)
        num = rank[inv.ravel()].reshape(gid.shape)
        self.nnode = first.size
        free = np.ones((self.nnode, 3), bool)
        on = {0: (K == 0) | (I == 0) | (I == 2 * nx), 1: (K == 0) | (J == 0) | (J == 2 * ny),
              2: K == 0}
        for c, m in on.items():
            free[num[m], c] = False
        gdof = np.where(free.ravel(), np.cumsum(free.ravel()), 0).reshape(-1, 3)
        self.neq = int(free.sum())
        self.num = num
        self.gdof = torch.as_tensor(gdof[num].reshape(len(num), 81), device=dev)
        xc = torch.as_tensor(mesh.coord[mesh.conn - 1], device=dev)  # (E, 8, 3)
        pts = np.stack([_G[li], _G[lj], _G[lk]], 1)                   # (27, 3)
        one = 1 + pts[:, None, :] * _CORNER[None]
        dsh = np.stack([_CORNER[None, :, a] * np.prod(np.delete(one, a, 2), 2) / 8
                        for a in range(3)], 1)                        # (27, 3, 8)
        shp = np.prod(one, 2) / 8
        self.coord = torch.einsum("ig,egd->eid", torch.as_tensor(shp, device=dev), xc)
        jac = torch.einsum("iag,egb->eiab", torch.as_tensor(dsh, device=dev), xc)
        self.detw = torch.linalg.det(jac) * torch.as_tensor(_W[li] * _W[lj] * _W[lk], device=dev)
        dl = np.zeros((27, 3, 27))
        for i in range(27):
            for n in range(27):
                a, b = (li[i], lj[i], lk[i]), (li[n], lj[n], lk[n])
                for d in range(3):
                    if all(a[q] == b[q] for q in range(3) if q != d):
                        dl[i, d, n] = _D[a[d], b[d]]
        # (E, 27 points, 3, 27 nodes)
        self.der = torch.matmul(torch.linalg.inv(jac), torch.as_tensor(dl, device=dev))
        mat = torch.as_tensor(mesh.mat_id.astype(np.int64) - 1, device=dev)
        gam, ym, nu, *_ = (torch.as_tensor(a, device=dev) for a in mesh.material_arrays())
        self.mat, self.gam = mat, gam[mat]
        lam = (ym * nu / ((1 + nu) * (1 - 2 * nu)))[mat]
        mu = (ym / (2 * (1 + nu)))[mat]
        c = torch.zeros(len(num), 6, 6, dtype=torch.float64, device=dev)
        c[:, :3, :3] = lam[:, None, None]
        for q in range(3):
            c[:, q, q] += 2 * mu
            c[:, 3 + q, 3 + q] = mu
        self.c = c
        load = torch.zeros(len(num), 27, 3, dtype=torch.float64, device=dev)
        load[:, :, 2] = -self.detw * self.gam[:, None]
        self.ext = self.scatter(load.reshape(len(num), 81, 1))

    def b(self, e0, e1):
        """Strain-displacement matrices (e, 27, 6, 81) of a run of elements."""
        d = self.der[e0:e1]
        m = torch.zeros(d.shape[0], 27, 6, 27, 3, dtype=torch.float64, device=self.dev)
        for row, parts in enumerate((((0, 0),), ((1, 1),), ((2, 2),), ((0, 1), (1, 0)),
                                     ((1, 2), (2, 1)), ((2, 0), (0, 2)))):
            for comp, axis in parts:
                m[:, :, row, :, comp] = d[:, :, axis, :]
        return m.reshape(d.shape[0], 27, 6, 81)

    def runs(self):
        e = self.gdof.shape[0]
        return [(a, min(e, a + 1024)) for a in range(0, e, 1024)]

    def matrices(self):
        self.k = torch.empty(self.gdof.shape[0], 81, 81, dtype=torch.float64, device=self.dev)
        for a, z in self.runs():
            b = self.b(a, z)
            cb = torch.matmul(self.c[a:z, None], b) * self.detw[a:z, :, None, None]
            self.k[a:z] = torch.bmm(b.reshape(z - a, 162, 81).transpose(1, 2).contiguous(),
                                    cb.reshape(z - a, 162, 81))
        d = torch.diagonal(self.k, dim1=1, dim2=2)
        self.diag = self.scatter(d[:, :, None])
        self.dinv = 1 / self.diag
        self.dinv[0] = 0
        return self

    def gather(self, x):
        return x[self.gdof]

    def scatter(self, y):
        """Sums of element vectors (E, 81, columns) at their equations: each
        equation's few places are gathered one after another."""
        if self.places is None:
            flat = self.gdof.reshape(-1)
            order = torch.argsort(flat, stable=True)
            count = torch.bincount(flat, minlength=self.neq + 1)
            begin = torch.cumsum(count, 0) - count
            self.places = []
            for k in range(int(count[1:].max())):
                here = k < count
                here[0] = False
                self.places.append((here[:, None], order[torch.where(here, begin + k, 0)]))
        y = y.reshape(-1, y.shape[2])
        out = torch.zeros(self.neq + 1, y.shape[1], dtype=torch.float64, device=self.dev)
        for here, at in self.places:
            out += torch.where(here, y[at], 0.0)
        return out

    def solve(self, f, x, tol, cap):
        """Jacobi-CG on every column of f from x, to |alpha| max|p| / max|x|
        <= tol or `cap` iterations."""
        r = f - self.scatter(torch.bmm(self.k, self.gather(x)))
        z = self.dinv * r
        p, rz, x = z.clone(), (r * z).sum(0), x.clone()
        for it in range(cap):
            kp = self.scatter(torch.bmm(self.k, self.gather(p)))
            alpha = rz / (p * kp).sum(0)
            alpha = torch.where(torch.isfinite(alpha), alpha, torch.zeros_like(alpha))
            x = x + alpha * p
            step = (alpha.abs() * p.abs().amax(0) / x.abs().amax(0)) if it % 8 == 7 else None
            r = r - alpha * kp
            z = self.dinv * r
            new = (r * z).sum(0)
            beta = new / rz
            p, rz = z + torch.where(torch.isfinite(beta), beta, torch.zeros_like(beta)) * p, new
            if step is not None and tol > 0 and float(step.max()) <= tol:
                break
        return x

    def body(self, x, t, st, ev, final):
        """One pass of the viscoplastic Mohr-Coulomb update of a trial at
        every Gauss point: (body load, effective stress, plastic strain, f)."""
        m = {k: torch.as_tensor(np.asarray(t[k]), device=self.dev)[self.mat][:, None]
             for k in ("phif", "cohf", "psif")}
        eps = torch.empty_like(ev)
        u = self.gather(x)
        for a, z in self.runs():
            eps[a:z] = torch.matmul(self.b(a, z), u[a:z, None, :, None])[..., 0]
        eff = torch.matmul(self.c[:, None], (eps - ev)[..., None])[..., 0] + st
        rad = math.pi / 180
        s1, s2, s3, s4, s5, s6 = eff.unbind(-1)
        sm = (s1 + s2 + s3) / 3
        j2 = ((s1 - s2) ** 2 + (s2 - s3) ** 2 + (s3 - s1) ** 2) / 6 + s4 ** 2 + s5 ** 2 + s6 ** 2
        j2 = j2.clamp(min=1e-12)
        d1, d2, d3 = s1 - sm, s2 - sm, s3 - sm
        j3 = d1 * d2 * d3 - d1 * s5 ** 2 - d2 * s6 ** 2 - d3 * s4 ** 2 + 2 * s4 * s5 * s6
        sq3 = math.sqrt(3)
        dsb = sq3 * j2.sqrt()
        th = torch.asin((-3 * sq3 * j3 / (2 * j2 ** 1.5)).clamp(-1, 1)) / 3
        sp, cp = torch.sin(m["phif"] * rad), torch.cos(m["phif"] * rad)
        f = sp * sm + dsb * (torch.cos(th) / sq3 - torch.sin(th) * sp / 3) - m["cohf"] * cp
        pl = f >= 0
        ss = torch.sin(m["psif"] * rad)
        sn, cn = torch.sin(th), torch.cos(th)
        t3, tn = torch.tan(3 * th), torch.sin(th) / torch.cos(th)
        edge = sn.abs() > 0.49
        q2 = torch.where(edge, (sq3 / 2 - torch.sign(sn) * ss / (2 * sq3)) * sq3 / 2 / dsb,
                         sq3 * cn / dsb * (1 + tn * t3 + ss * (t3 - tn) / sq3) / 2)
        q3 = torch.where(edge, torch.zeros_like(th),
                         1.5 * (sq3 * sn + ss * cn) / (torch.cos(3 * th) * dsb * dsb))
        # gradients of the invariants with respect to the stress
        one = torch.zeros_like(eff)
        one[..., :3] = 1.0
        dev = torch.stack([d1, d2, d3, 2 * s4, 2 * s5, 2 * s6], -1)
        sq = torch.stack([d1 * d1 + s4 * s4 + s6 * s6, d2 * d2 + s4 * s4 + s5 * s5,
                          d3 * d3 + s5 * s5 + s6 * s6, 2 * (d1 * s4 + s4 * d2 + s6 * s5),
                          2 * (s4 * s6 + d2 * s5 + s5 * d3),
                          2 * (d1 * s6 + s4 * s5 + s6 * d3)], -1)
        g3 = sq - one * (2.0 / 3.0) * j2[..., None]
        dq = one / 3 * ss[..., None] + dev * q2[..., None] + g3 * q3[..., None]
        evp = torch.where(pl[..., None], f[..., None] * dq * t["dt"], torch.zeros_like(dq))
        ev = ev + evp
        load = None
        if not final:
            w = torch.matmul(self.c[:, None], evp[..., None])[..., 0] * self.detw[..., None]
            le = torch.empty(self.gdof.shape[0], 81, 1, dtype=torch.float64, device=self.dev)
            for a, z in self.runs():
                le[a:z] = torch.bmm(self.b(a, z).reshape(z - a, 162, 81).transpose(1, 2).contiguous(),
                                    w[a:z].reshape(z - a, 162, 1))
            load = self.scatter(le)[:, 0]
        return load, eff, ev, f

    def zeros(self):
        return torch.zeros(self.gdof.shape[0], 27, 6, dtype=torch.float64, device=self.dev)


def _host(t):
    return t.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch" and case["ncol"] * case["nx"] * case["ny"] * case["nz"] > 1_000_000:
        return None  # about a minute
    p = _Plain(case, seed)
    if kind == "setup":
        p.matrices()
        xyz = np.empty((p.nnode, 3))
        xyz[p.num.ravel()] = _host(p.coord).reshape(-1, 3)
        return {"extload": _host(p.ext[:, 0]), "dinv": _host(p.dinv[:, 0]), "gdof_elmt": None,
                "g_coord": xyz}
    if kind == "stage":
        x = np.random.default_rng([seed, 5]).normal(0, 1e-2, p.neq + 1)
        x[0] = 0.0
        u = p.gather(torch.as_tensor(x, device=p.dev))
        sig = torch.as_tensor(_stress0(case, p.mesh, seed), device=p.dev)
        st, le = p.zeros(), torch.empty(len(p.mat), 81, 1, dtype=torch.float64, device=p.dev)
        for a, z in p.runs():
            b = p.b(a, z)
            st[a:z] = torch.matmul(p.c[a:z, None], torch.matmul(b, u[a:z, None, :, None]))[..., 0]
            w = sig[a:z] * p.detw[a:z, :, None]
            le[a:z] = torch.bmm(b.reshape(z - a, 162, 81).transpose(1, 2).contiguous(),
                                w.reshape(z - a, 162, 1))
        return {"stress": _host(st), "load": _host(p.scatter(le)[:, 0] - p.ext[:, 0])}
    p.matrices()
    if kind in ("dropin", "solve"):
        zero = torch.zeros_like(p.ext)
        if case["cap"]:  # the iterate that many iterations reach
            return {"u": _host(p.solve(p.ext, zero, 0.0, case["cap"])[:, 0])}
        return {"u": _host(p.solve(p.ext, zero, 2e-14, MAXITER)[:, 0])}
    xel = p.solve(p.ext, torch.zeros_like(p.ext), 2e-14, MAXITER)
    strengths = _strengths(case, p.mesh, seed)
    if kind == "plastic":
        t = _factored(case, p.mesh, strengths[0], case["srf"])
        load, _, ev, _ = p.body(xel[:, 0], t, p.zeros(), p.zeros(), False)
        x = p.solve(p.ext + load[:, None], xel, 2e-14, MAXITER)
        _, eff, ev, f = p.body(x[:, 0], t, p.zeros(), ev, True)
        return {"x": _host(x[:, 0]), "bodyload": _host(load), "evpt": _host(ev),
                "stress": _host(eff), "flags": None, "fmax": float(f.max().clamp(min=0)),
                "sig": None, "psigma": None, "nsigma": None}
    if kind == "batch":
        trials = [_factored(case, p.mesh, t, case["srf"]) for t in strengths]
        first = [p.body(xel[:, 0], t, p.zeros(), p.zeros(), False) for t in trials]
        f = p.ext + torch.stack([q[0] for q in first], 1)
        x = p.solve(f, xel.expand(-1, len(trials)).contiguous(), 2e-14, MAXITER)
        fm = [float(p.body(x[:, j], t, p.zeros(), first[j][2], True)[3].max().clamp(min=0))
              for j, t in enumerate(trials)]
        return {"x": _host(x.T.contiguous()), "flags": None, "fmax": np.array(fm)}
    out = []
    for s in strengths:
        for srf in (0.8, 0.9):
            t = _factored(case, p.mesh, s, srf)
            x = old = xel
            ev, body = p.zeros(), torch.zeros_like(xel)
            for it in range(1, 13):
                if it > 1:
                    x = p.solve(p.ext + body, x, 2e-14, MAXITER)
                conv = it > 1 and float((x - old).abs().max() / x.abs().max()) <= NL_TOL
                old = x
                if conv or it == 12:
                    break
                load, _, ev, _ = p.body(x[:, 0], t, p.zeros(), ev, False)
                body = body + load[:, None]
            if it == 12:  # the sweep ends at its first failing factor
                break
        out.append(_host(x[:, 0]))
    return {"x": np.stack(out)}
