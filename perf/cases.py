"""Performance cases of the engine: what a micromagnetic program has it do, through the public entry
points of feellgood_amd.engine, from the smallest meshes to the 2M-tetrahedron film.

A case of kind
  run     is a stretch of a simulation between two saves: set_state, the first demag potentials, a
          number of steps of the loop body (Engine.step), get_state;
  field   is the same under a space-dependent applied field, through the separate calls;
  batch   is the same for independent nanodots side by side in one context (Engine.batch);
  spin    is one spin-accumulation solve at a magnetization (SpinSolver.solve);
  train   is one training batch of the learned initial guess: a solve that records its features,
          then the forward pass, the backward pass and the weight gradients (guess_gradient).
Meshes, textures, applied fields, basis angles and network weights are seeded.
"""
import ctypes as C
import math

import numpy as np
import torch

from feellgood_amd import native as nv
from feellgood_amd.engine import Engine, SpinSolver
from feellgood_amd.mesh import HostMesh
from feellgood_amd.workloads import MU0, build_dots, dots_workload, guess_weights_path, prefactor

GAMMA0 = 1.76085962784e11 * MU0
THETA = 0.5
TOL = 1e-10

# a run's fields and their defaults: shape and cells of the mesh, cell size [nm], jitter, material,
# step, demag method and precision, Krylov form, trained guess, steps between two saves
RUN = dict(kind="run", shape="cuboid", nx=1, ny=1, nz=1, h=3.0, jitter=0.1, alpha=0.1, K=0.0, dt=5e-14, demag="fmm",
           order=8, leaf=64, precision="fp64", krylov="fp64", guess=False, steps=10)


def _run(name, **kw):
    c = dict(RUN, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a unit-test-sized block with the default (exact) demag: the call and launch overheads of a step
        _run("block exact", nx=8, ny=6, nz=2, h=5.0, K=1e4, demag="direct"),
        # an ellipsoid of the size of the reference's own end-to-end example, exact demag
        _run("ellipsoid exact", shape="ellipsoid", nx=10, ny=8, nz=6, h=4.0, demag="direct", dt=2e-14),
        # the 100 nm cube of the benchmark (48,000 tetrahedra), FMM demag in FP64
        _run("cube", nx=20, ny=20, nz=20, h=5.0, jitter=0.0, alpha=0.5, dt=1e-13),
        # a small film whose exact demag is still affordable: the accuracy reference of a study
        _run("film exact", nx=48, ny=32, nz=3, demag="direct"),
        # a mid-size film in the fast configuration: trained guess and mixed-precision FMM
        _run("film 220k fast", nx=111, ny=56, nz=6, alpha=0.02, precision="mixed", guess=True),
        # the plain FP64 FMM configuration on a film of odd sizes
        _run("film 490k fp64", nx=167, ny=83, nz=6, alpha=0.02, steps=6),
        # the headline: 2M tetrahedra, trained guess and mixed-precision FMM
        _run("film 2M fast", nx=333, ny=167, nz=6, h=3.0, alpha=0.02, precision="mixed", guess=True),
        # a wire (domain-wall geometry): deep octree, many empty cells; mixed precision in the FMM and
        # in the Krylov loop
        _run("wire mixed", shape="wire", nx=10, ny=10, nz=150, h=5.0, alpha=0.05, dt=2e-14, precision="mixed",
             krylov="mixed"),
        # a space-dependent field (an antenna or a tip), through the separate calls
        _run("gradient field", kind="field", nx=61, ny=40, nz=4),
        # a parameter sweep over nanodots in one context, each with its own solve
        dict(name="dots 64", kind="batch", count=64, h=4.5, leaf=128, block=1024, steps=10),
        # the spin accumulation of a current-driven bar, solved once per step of such a run
        dict(name="spin bar", kind="spin", nx=40, ny=10, nz=8, h=2.0),
        # a training batch of the learned guess on a film
        dict(name="guess training", kind="train", nx=100, ny=50, nz=3, h=3.0),
    ]


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def _film_cells(rng, nodes):
    """Cells of a film or block of about that many nodes, odd sizes included."""
    nz = rng.choice([2, 3, 4, 5, 6, 9])
    n = max(nodes / (nz + 1), 9.0)
    r = rng.uniform(1.0, 3.0)
    return dict(nx=max(2, round(math.sqrt(n * r)) - 1), ny=max(2, round(math.sqrt(n / r)) - 1), nz=nz)


def draw(rng):
    k = rng.random()
    if k < 0.22:  # exact demag: up to a few thousand nodes
        return _run("", **_film_cells(rng, _log(rng, 150, 9000)), h=round(rng.uniform(2.0, 5.0), 2), demag="direct",
                    alpha=rng.choice([0.02, 0.1, 0.5]), K=rng.choice([0.0, 2e4]))
    if k < 0.62:  # FMM demag, either precision
        mixed = rng.random() < 0.5
        return _run("", **_film_cells(rng, _log(rng, 2000, 120000)), h=round(rng.uniform(2.0, 4.0), 2),
                    alpha=rng.choice([0.02, 0.1, 0.5]), K=rng.choice([0.0, 2e4]), leaf=rng.choice([32, 64, 64, 128]),
                    order=rng.choice([6, 8, 8, 8]), precision="mixed" if mixed else "fp64",
                    krylov="mixed" if mixed and rng.random() < 0.3 else "fp64", guess=mixed and rng.random() < 0.5)
    if k < 0.72:
        n = rng.randint(5, 9)
        return _run("", shape="wire", nx=n, ny=n, nz=round(_log(rng, 30, 160)), h=5.0, alpha=0.05, dt=2e-14,
                    precision=rng.choice(["fp64", "mixed"]))
    if k < 0.80:
        return _run("", kind="field", **_film_cells(rng, _log(rng, 2000, 40000)), precision=rng.choice(["fp64", "mixed"]))
    if k < 0.88:
        return dict(kind="batch", count=round(_log(rng, 4, 64)), h=round(rng.uniform(4.5, 6.0), 2), leaf=128,
                    block=rng.choice([256, 512, 1024]), steps=10)
    if k < 0.94:
        return dict(kind="spin", nx=round(_log(rng, 10, 60)), ny=rng.randint(3, 10), nz=rng.randint(3, 10), h=2.0)
    return dict(kind="train", **_film_cells(rng, _log(rng, 2000, 60000)), h=3.0)


# ---------------------------------------------------------------------- inputs

def _lengths(c):
    return tuple(c["h"] * c[k] for k in ("nx", "ny", "nz"))


def _mesh(c, seed):
    """A prepared mesh of the case: jittered cuboid, ellipsoid or cylinder."""
    shape = c.get("shape", "cuboid")
    if shape == "ellipsoid":
        m = HostMesh.ellipsoid((0.0, 0.0, 0.0), tuple(0.5 * v for v in _lengths(c)), 0.5 * c["h"])
    elif shape == "wire":
        m = HostMesh.cylinder((0.0, 0.0), 0.0, 0.5 * c["h"] * c["nx"], c["h"] * c["nz"], c["h"])
    else:
        m = HostMesh.cuboid(_lengths(c), (c["nx"], c["ny"], c["nz"]), jitter=c.get("jitter", 0.1), seed=seed % 65521)
    m.prepare({"volume": dict(Ms=8e5, Ae=1.3e-11, alpha=c.get("alpha", 0.1), K=c.get("K", 0.0), uk=(0.0, 1.0, 0.0))})
    return m


def _unit(u):
    return u / np.linalg.norm(u, axis=1, keepdims=True)


def _texture(pos, rng, wire=False):
    """A smooth, nearly single-domain texture (an S-state of seeded amplitude and a slow ripple): along
    x in films and blocks, along the axis with a reversed end domain in wires."""
    lo, hi = pos.min(0), pos.max(0)
    s = (pos - lo) / (hi - lo).max()
    ph = rng.uniform(0.15, 0.4) * np.sin(np.pi * s[:, 0] / s[:, 0].max())
    rip = 0.02 * np.sin(2 * np.pi * (s @ rng.uniform(0.5, 2.0, 3)) + rng.uniform(0, 6))
    if wire:
        u = np.stack([rip, 0.02 * np.cos(2 * np.pi * s[:, 2]), np.where(s[:, 2] < 0.05, -1.0, 1.0)], axis=1)
    else:
        u = np.stack([np.cos(ph), np.sin(ph), rip], axis=1)
    return _unit(u)


def _field(rng):
    """Applied field of 20-40 mT, roughly against the texture, in A/m."""
    a, t = math.radians(rng.uniform(150.0, 190.0)), rng.uniform(-0.1, 0.1)
    return np.array([math.cos(a), math.sin(a), t]) * rng.uniform(0.02, 0.04) / MU0


def _inputs(c, seed):
    """Everything of a case but the handles: meshes, texture, field, basis angles, and what else its kind takes."""
    rng = np.random.default_rng(seed)
    s = dict(case=c)
    if c["kind"] == "batch":
        w = dict(dots_workload(), h=c["h"])
        s["meshes"], u = build_dots(w, c["count"])
        s["u"], s["dt"] = _unit(rng.normal(size=u.shape)), w["dt"]
    elif c["kind"] == "spin":
        s["meshes"] = [_mesh(c, seed)]
        pos = s["meshes"][0].arrays()["pos"]
        s["bar"] = _bar(s["meshes"][0])
        s["u"] = _texture(pos, rng)
        s["V"] = -1e6 * rng.uniform(0.5, 2.0) * (pos[:, 0] - pos[:, 0].min())
        return s
    else:
        s["meshes"] = [_mesh(c, seed)]
        s["u"] = _texture(s["meshes"][0].arrays()["pos"], rng, c.get("shape") == "wire")
        s["dt"] = c.get("dt", 5e-14)
    s["H"] = _field(rng)
    s["r"] = rng.uniform(0.0, 2.0 / math.pi, c.get("steps", 1))
    if c["kind"] == "field":
        # amplitude over the steps, and a Gaussian spot of field over a gradient at the Gauss points
        m = s["meshes"][0].mesh
        pg = np.zeros(15 * m.n_tets)
        nv.hip_lib().fg_gauss_points(C.byref(m), nv.dptr(pg))
        pg = pg.reshape(-1, 5, 3)
        q = (pg - pg.min((0, 1))) / (pg.max((0, 1)) - pg.min((0, 1)))
        spot = np.exp(-((q - rng.uniform(0.3, 0.7, 3)) ** 2).sum(-1) / 0.05)
        s["space"] = spot[..., None] * s["H"] + q * np.array([5e3, -3e3, 1e3])
        s["amp"] = rng.uniform(0.5, 1.0, c["steps"])
    if c["kind"] == "train":
        n = len(s["u"])
        v = rng.normal(size=(n, 3)) * 2e9 + GAMMA0 * np.cross(s["u"], s["H"])
        s["v"] = v - np.sum(v * s["u"], axis=1, keepdims=True) * s["u"]
        s["phi"], s["phiv"] = rng.normal(size=n) * 1e-4, rng.normal(size=n) * 1e5
        p = rng.normal(size=nv.FG_GUESS_NPARAM) * 0.15
        p[-nv.FG_GUESS_NSCALE:] = [1 / 3e4, 1 / 2e9, 5e8, 1 / 1e7]
        s["params"] = p.astype(np.float32)
    return s


NAN = float("nan")
SPIN_VOL = dict(sigma=5e6, N0=1e47, P=0.4, lsd=5e-9, lsf=10e-9)
SPIN_S, SPIN_JN, SPIN_UP = (2e6, -1e6, 5e5), 3e10, (0.0, 0.6, 0.8)


def _bar(hm):
    """The mesh as a bar whose right half is magnetic, with the surface regions left end, right end
    and the rest: (fg_mesh view, the arrays that it points to)."""
    a = hm.arrays()
    pos, tets, tris = (np.ascontiguousarray(a[k]) for k in ("pos", "tets", "tris"))
    x0, x1 = pos[:, 0].min(), pos[:, 0].max()
    treg = (pos[tets].mean(axis=1)[:, 0] > 0.5 * (x0 + x1)).astype(np.int32)
    tx = pos[tris][:, :, 0]
    freg = np.full(len(tris), 2, np.int32)
    freg[np.all(tx < x0 + 1e-6 * (x1 - x0), axis=1)] = 0
    freg[np.all(tx > x1 - 1e-6 * (x1 - x0), axis=1)] = 1
    dms = np.zeros(len(tris))
    vol, surf = (nv.VolumeRegion * 2)(), (nv.SurfaceRegion * 3)()
    vol[0].Ms, vol[1].Ms = 0.0, 8e5
    m = nv.Mesh()
    m.n_nodes, m.n_tets, m.n_tris, m.n_vol_regions, m.n_surf_regions = len(pos), len(tets), len(tris), 2, 3
    m.pos, m.tri_dMs = (x.ctypes.data_as(C.POINTER(C.c_double)) for x in (pos, dms))
    m.tet_nodes, m.tet_region, m.tri_nodes, m.tri_region = (x.ctypes.data_as(C.POINTER(C.c_int32))
                                                            for x in (tets, treg, tris, freg))
    m.vol, m.surf = C.cast(vol, C.POINTER(nv.VolumeRegion)), C.cast(surf, C.POINTER(nv.SurfaceRegion))
    return m, (hm, pos, tets, tris, treg, freg, dms, vol, surf)


def prepare(case, seed):
    c = case
    s = _inputs(c, seed)
    if c["kind"] == "spin":
        vol = [nv.SpinVolume(*(SPIN_VOL[k] for k in ("sigma", "N0", "P", "lsd", "lsf")))] * 2
        d3 = C.c_double * 3
        surf = [nv.SpinSurface(NAN, d3(NAN, NAN, NAN), d3(*SPIN_S)), nv.SpinSurface(SPIN_JN, d3(*SPIN_UP), d3(NAN, NAN, NAN)),
                nv.SpinSurface(NAN, d3(NAN, NAN, NAN), d3(NAN, NAN, NAN))]
        s["solver"] = SpinSolver(s["bar"][0], vol, surf, s["V"], tol=1e-8, max_iter=2000)
        return s
    kw = dict(tol=TOL, max_iter=1000)
    if c["kind"] == "batch":
        s["engine"] = Engine.batch([m.mesh for m in s["meshes"]], demag="fmm", precision="mixed", fmm_leaf=c["leaf"],
                                   batch_solver="persistent", batch_block=c["block"], **kw)
        return s
    m = s["meshes"][0].mesh
    if c["kind"] == "train":
        s["engine"] = e = Engine(m, demag="direct", **kw)
        e.guess_init(0)
        e.guess_set(s["params"])
        return s
    s["engine"] = e = Engine(m, demag=c["demag"], fmm_order=c["order"], fmm_leaf=c["leaf"], precision=c["precision"],
                             krylov=c["krylov"], **kw)
    if c["guess"]:
        path = guess_weights_path("film")
        e.guess_set(np.load(path))
        e.guess_enable()
    if c["kind"] == "field":
        e.set_space_field(s["space"])
    return s


# ---------------------------------------------------------------------- one pass

def run(state):
    s = state
    c = s["case"]
    if c["kind"] == "spin":
        acc, info = s["solver"].solve(s["u"], accumulate=False)
        return dict(s=acc)
    e, dt = s["engine"], s["dt"]
    pref = prefactor(dt)
    if c["kind"] == "train":
        e.set_state(nv.FG_BOTH, u=s["u"], v=s["v"], phi=s["phi"], phiv=s["phiv"])
        e.base_projection(s["r"][0])
        e.prepare_elements(s["H"], dt, pref)
        failed, info = e.solve(dt)
        if failed:
            raise RuntimeError("the solve failed")
        grad, loss, ref = e.guess_gradient()
        return dict(grad=grad, loss=loss, loss_ref=ref, features=e.guess_features()[:, :9])
    e.set_state(nv.FG_BOTH, u=s["u"])
    e.calc_demag()
    e.evolution()
    E = angle = None
    for k, r in enumerate(s["r"]):
        if c["kind"] == "field":
            e.base_projection(r)
            e.prepare_elements_amp(s["amp"][k], dt, pref)
            failed, info = e.solve(dt)
            if failed:
                raise RuntimeError("the solve failed")
            e.calc_demag()
            E = e.energy_amp(s["amp"][k])
            e.evolution()
            angle = e.max_angle()
        else:
            rc, info, E, angle = e.step(r, s["H"], dt, pref)
            if rc != nv.FG_OK:
                raise RuntimeError(f"the step was not taken: {rc}")
    u, v, phi, phiv = e.get_state(nv.FG_CURRENT)
    return dict(u=u, v=v, phi=phi, phiv=phiv, E=E, angle=angle)


# ---------------------------------------------------------------------- work and tolerance

def _sizes(c):
    """Nodes, tetrahedra and surface triangles of the case (the batch's are those of mean dots)."""
    if c["kind"] == "batch":
        v = 4 / 3 * math.pi * 35.0 * 35.0 * 11.5 * c["count"] / c["h"] ** 3
        return v * 1.5, v * 6, v * 2.5
    x, y, z = c["nx"], c["ny"], c["nz"]
    if c.get("shape") == "ellipsoid":
        x, y, z = 1.6 * x, 1.6 * y, 1.6 * z
    if c.get("shape") == "wire":
        x, y = 0.89 * x, 0.89 * y
    return (x + 1) * (y + 1) * (z + 1), 6 * x * y * z, 4 * (x * y + y * z + z * x)


def work(case):
    c = case
    N, T, F = _sizes(c)
    if c["kind"] == "spin":
        it = 60  # iterations of a stencil product pair over 3 N unknowns
        return dict(bytes=T * 16 + N * 24 * 3 + it * 2 * (15 * N * 12 + 3 * N * 8 * 6), flops=it * 2 * 15 * N * 6)
    if c["kind"] == "train":
        return dict(bytes=N * (128 + 64 + 24) + T * 152 + 10 * (15 * N * 12 + 16 * N * 12),
                    flops=N * 6 * (24 * 64 + 64 * 64 + 64 * 3) + 400 * T)
    # a step: the element pass, the stencil products of a few iterations, the demag potentials of u and v
    # and the energies; geometry, stencil and states read once per use, results written once
    step_bytes = 3 * T * 152 + 9 * (15 * N * 12) + 30 * N * 64
    step_flops = 900 * T + 9 * 15 * N * 6
    src, n_demag = 5 * T + 4 * F, c["steps"] + 1
    if c.get("demag") == "direct":
        demag_bytes, demag_flops = src * 40 + N * 40, N * src * 14
    else:
        # an order-8 FMM: 2 x 81 coefficients per source and per target, near sources by pairs
        demag_bytes, demag_flops = src * 16 + N * 40, 2 * 81 * 2 * (src + N * 60) + N * 27 * 64 * 6
    return dict(bytes=c["steps"] * step_bytes + n_demag * demag_bytes + N * 8 * 11,
                flops=c["steps"] * step_flops + n_demag * demag_flops)


def tolerance(case):
    """About four times the largest error over the outputs against exact(): the Krylov tolerances where
    everything else is exact, FP32 sums in the training pass, and the multipole truncation (largest in
    the potential of v, whose far field the mixed-precision FMM takes to degree 4)."""
    c = case
    if c["kind"] == "spin":
        return dict(rel=4e-7, max=4e-6)
    if c["kind"] == "train":
        return dict(rel=1e-6, max=1e-5)
    if c["kind"] == "batch":
        return dict(rel=1e-2, max=0.2)
    if c["demag"] == "direct":
        return dict(rel=1e-8, max=4e-7)
    if c["order"] < 8:
        return dict(rel=2e-3, max=2e-2)
    return dict(rel=1e-3, max=1e-2) if c["precision"] == "mixed" else dict(rel=2e-4, max=4e-3)


# ---------------------------------------------------------------------- 64-bit results

DEV = "cuda"
F64 = torch.float64
TET_A = np.array([[.25, .25, .25, .25], [.5, 1 / 6, 1 / 6, 1 / 6], [1 / 6, 1 / 6, 1 / 6, .5], [1 / 6, 1 / 6, .5, 1 / 6],
                  [1 / 6, .5, 1 / 6, 1 / 6]])
TET_W = np.array([-2 / 15, 3 / 40, 3 / 40, 3 / 40, 3 / 40])
TRI_A = np.array([[1 / 3, 1 / 3, 1 / 3], [.6, .2, .2], [.2, .6, .2], [.2, .2, .6]])
TRI_W = np.array([-27 / 96, 25 / 96, 25 / 96, 25 / 96])


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), device=DEV)


def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


def _gradients(X):
    """P1 gradients [T, 4, 3] and Jacobian determinants [T] of tetrahedra with vertices X [T, 4, 3]."""
    J = X[:, 1:] - X[:, :1]
    g = torch.linalg.inv(J).transpose(1, 2)
    return torch.cat([-g.sum(1, keepdim=True), g], dim=1), torch.linalg.det(J)


def _bicgstab(A, b, x, D, tol):
    """x with ||b - A x|| near tol ||b||: BiCGSTAB with the preconditioner D, restarted from the true residual at each 1e-5 of it."""
    last = math.inf
    for _ in range(12):
        r = b - A(x)
        start = float(r.norm())
        if start <= tol * float(b.norm()) or start > 0.5 * last:  # there, or at the rounding of b - A x
            break
        last = start
        r = r / start
        rt, p, v, d = r.clone(), torch.zeros_like(r), torch.zeros_like(r), torch.zeros_like(r)
        rho = al = om = 1.0
        for _ in range(300):
            rho1 = float((rt * r).sum())
            p = r + (rho1 / rho) * (al / om) * (p - om * v)
            rho, ph = rho1, D(p)
            v = A(ph)
            rv = float((rt * v).sum())
            if rv == 0.0 or om == 0.0:
                break
            al = rho / rv
            s = r - al * v
            sh = D(s)
            t = A(sh)
            tt = float((t * t).sum())
            om = float((t * s).sum()) / tt if tt > 0.0 else 0.0
            d = d + al * ph + om * sh
            r = s - om * t
            if float(r.norm()) <= 1e-5:
                break
        x = x + start * d
    return x


class _Llg:
    """The weak LLG step of the reference in 64 bits on torch: lumped mass with the effective damping,
    exchange stencil, applied, anisotropy and demag fields; exact demag potentials by summation over the
    Gauss points with the analytic self terms of the surface triangles."""

    def __init__(self, meshes):
        pos, tets, tris, dms, par = [], [], [], [], []
        self.inst = []  # node, tetrahedron and triangle ranges of the instances
        n = t = f = 0
        for hm in meshes:
            a, m = hm.arrays(), hm.mesh
            pos.append(a["pos"])
            tets.append(a["tets"] + n)
            tris.append(a["tris"] + n)
            dms.append(a["dMs"])
            v = m.vol[0]
            par.append(np.tile([v.alpha, v.Ae, v.Ms, v.K, *v.uk], (len(a["tets"]), 1)))
            self.inst.append((n, n + len(a["pos"]), t, t + len(a["tets"]), f, f + len(a["tris"])))
            n, t, f = self.inst[-1][1::2]
        self.pos, self.tets, self.tris = _t(np.concatenate(pos)), _t(np.concatenate(tets)).long(), _t(np.concatenate(tris)).long()
        self.dms, par = _t(np.concatenate(dms)), _t(np.concatenate(par))
        self.alpha, self.Ae, self.Ms, self.K = (par[:, k:k + 1] for k in range(4))
        self.uk = par[:, 4:7]
        self.N = n
        self.ga, self.ta = _t(TET_A), _t(TRI_A)
        X = self.pos[self.tets]
        self.da, det = _gradients(X)
        self.w = det[:, None] * _t(TET_W)
        P = self.pos[self.tris]
        cr = torch.linalg.cross(P[:, 1] - P[:, 0], P[:, 2] - P[:, 0])
        self.surf = 0.5 * cr.norm(dim=1, keepdim=True)
        self.nrm = cr / cr.norm(dim=1, keepdim=True)
        self.tw = 2 * self.surf * _t(TRI_W)
        self.P = P
        self.tgauss = torch.einsum("ga,tak->tgk", self.ga, X)
        self.fgauss = torch.einsum("ga,tak->tgk", self.ta, P)
        self.Abis = 2 * self.Ae / (MU0 * self.Ms)
        self.Kbis = 2 * self.K / (MU0 * self.Ms)
        self.mass = self._nodes((self.w @ self.ga)[..., None])
        self.Ke = self.Abis[:, :, None] * self.w.sum(1)[:, None, None] * (self.da @ self.da.transpose(1, 2))
        self.sd = self._nodes(torch.diagonal(self.Ke, dim1=1, dim2=2)[..., None])
        e = torch.cat([self.tets[:, [i, j]] for i in range(4) for j in range(i + 1, 4)])
        self.edges = e

    def _nodes(self, x):
        """Sums [N, k] of element contributions x [T, 4, k]."""
        return torch.zeros(self.N, x.shape[-1], dtype=F64, device=DEV).index_add_(0, self.tets.reshape(-1), x.reshape(-1, x.shape[-1]))

    def potentials(self, *fields):
        """phi [N] of each field [N, 3]."""
        qt = [-self.Ms * self.w * (self.da * u[self.tets]).sum((1, 2))[:, None] for u in fields]
        sn = [(u[self.tris] * self.nrm[:, None]).sum(-1) for u in fields]
        qf = [self.dms[:, None] * self.tw * (s @ self.ta.T) for s in sn]
        phi = [torch.zeros(self.N, dtype=F64, device=DEV) for _ in fields]
        for n0, n1, t0, t1, f0, f1 in self.inst:
            y = torch.cat([self.tgauss[t0:t1].reshape(-1, 3), self.fgauss[f0:f1].reshape(-1, 3)]).T.contiguous()
            q = [torch.cat([a[t0:t1].reshape(-1), b[f0:f1].reshape(-1)]) for a, b in zip(qt, qf)]
            step = max(1, int(6e7) // y.shape[1])
            for a in range(n0, n1, step):
                x = self.pos[a:min(a + step, n1)]
                r2 = (x[:, 0:1] - y[0]).square_()
                for k in (1, 2):
                    d = x[:, k:k + 1] - y[k]
                    r2.addcmul_(d, d)
                r2.rsqrt_()
                for p, c in zip(phi, q):
                    p[a:a + len(x)] = torch.mv(r2, c)
        # the triangles' own vertices: the Gauss-point sum is replaced by the analytic potential
        for i in range(3):
            j, k = (i + 1) % 3, (i + 2) % 3
            a, b = self.P[:, j] - self.P[:, i], self.P[:, k] - self.P[:, i]
            bl = a.norm(dim=1)
            tt = (a * b).sum(1) / bl
            s2 = 2 * self.surf[:, 0]
            h = s2 / bl
            c = (tt - bl) / h
            fc = torch.sqrt(1 + c * c)
            r = h * torch.sqrt(1 + (tt / h) ** 2)
            xi = bl * torch.log((c * tt + h + fc * r) / (bl * (c + fc))) / fc
            dist = (self.P[:, i:i + 1] - self.fgauss).norm(dim=2)
            for p, s, f in zip(phi, sn, qf):
                pot = xi * s[:, i] + ((xi * (h + c * tt) - bl * (r - bl)) * s[:, j] + bl * (r - bl - c * xi) * s[:, k]) * bl / (
                    s2 * (1 + c * c))
                p.index_add_(0, self.tris[:, i], 0.5 * self.dms * pot - (f / dist).sum(1))
        return [p / (4 * math.pi) for p in phi]

    def assemble(self, u, v, phi, phiv, H, dt):
        """(D [N, 1], F [N, 3]); H: a uniform field [3] or one per Gauss point [T, 5, 3]."""
        U, V = u[self.tets], v[self.tets]
        dU = self.da.transpose(1, 2) @ U                    # [T, k, 3]: gradient of u along k
        Hd = -(phi[self.tets][:, None] @ self.da)[:, 0]
        Hv = -(phiv[self.tets][:, None] @ self.da)[:, 0]
        Ug, Vg = self.ga @ U, self.ga @ V
        sdt = THETA * dt
        H0 = Hd[:, None] + H
        uk = self.uk[:, None]
        Han = self.Kbis[..., None] * _dot(uk, Ug + sdt * Vg) * uk
        uH = (-self.Abis * (dU * dU).sum((1, 2))[:, None] + self.Kbis * _dot(Ug, uk)[..., 0] ** 2 + _dot(Ug, H0)[..., 0])
        rdt, al = GAMMA0 * dt, self.alpha
        M = 2 * al * 0.1 / rdt
        ae = torch.where(uH > 0, al + rdt / 2 * torch.minimum(uH, M),
                         torch.where(uH < -M, al / (1 + rdt / (2 * al) * M), al / (1 - rdt / (2 * al) * uH)))
        Ht = H0 + Han + sdt * Hv[:, None]
        gex = self.da @ dU
        F = torch.einsum("ga,tg,tgk->tak", self.ga, self.w, Ht) - (self.w.sum(1)[:, None] * self.Abis)[..., None] * gex
        return self._nodes(((self.w * ae) @ self.ga)[..., None]), self._nodes(F)

    def solve(self, u, v, phi, phiv, H, dt):
        """The tangent solution x [N, 3] (v = gamma0 x) and the tangent right-hand side."""
        D, F = self.assemble(u, v, phi, phiv, H, dt)
        cst = prefactor(dt) * THETA * dt * GAMMA0

        def tangent(a):
            return a - _dot(a, u) * u

        def A(x):
            return tangent(D * x + self.mass * torch.linalg.cross(u, x) + cst * self._nodes(self.Ke @ x[self.tets]))

        d = D + cst * self.sd

        def node_block(y):  # the inverse of d + m [u]x on the tangent plane
            return tangent(d * y - self.mass * torch.linalg.cross(u, y)) / (d * d + self.mass * self.mass)

        b = tangent(F)
        return _bicgstab(A, b, tangent(v) / GAMMA0, node_block, 1e-13), b

    def energies(self, u, phi, H):
        U, p = u[self.tets], phi[self.tets]
        dU = self.da.transpose(1, 2) @ U
        Ug, pg = self.ga @ U, p @ self.ga.T
        div = torch.diagonal(dU, dim1=1, dim2=2).sum(1, keepdim=True)
        w = self.w
        ex = (self.Ae * w * (dU * dU).sum((1, 2))[:, None]).sum()
        an = -(self.K * w * _dot(Ug, self.uk[:, None])[..., 0] ** 2).sum()
        dm = -0.5 * MU0 * (self.Ms * w * div * pg).sum()
        ze = -MU0 * (self.Ms * w * (Ug * H).sum(-1)).sum()
        un = (u[self.tris] * self.nrm[:, None]).sum(-1) @ self.ta.T
        dm = dm + 0.5 * MU0 * (self.dms[:, None] * self.tw * un * (phi[self.tris] @ self.ta.T)).sum()
        return np.array([float(ex), float(an), float(dm), float(ze)])

    def angle(self, u):
        return math.acos(min(1.0, float((u[self.edges[:, 0]] * u[self.edges[:, 1]]).sum(1).min())))


def _exact_steps(s):
    c = s["case"]
    L = _Llg(s["meshes"])
    u, dt = _t(s["u"]), s["dt"]
    v = torch.zeros_like(u)
    phi, phiv = L.potentials(u, v)
    space = _t(s["space"]) if c["kind"] == "field" else None
    for k in range(c["steps"]):
        H = s["amp"][k] * space if space is not None else _t(s["H"])
        x, _ = L.solve(u, v, phi, phiv, H, dt)
        v = GAMMA0 * x
        u = u + dt * v
        u = u / u.norm(dim=1, keepdim=True)
        phi, phiv = L.potentials(u, v)
    return dict(u=u, v=v, phi=phi, phiv=phiv, E=L.energies(u, phi, H), angle=L.angle(u))


def _exact_spin(s):
    m, (hm, pos, tets, tris, treg, freg, *_rest) = s["bar"]
    q, mu_e = 1.602176634e-19, 6.62607015e-34 / (4 * math.pi * 9.1093837139e-31)
    p = SPIN_VOL
    D0 = 2 * p["sigma"] / (q * q * p["N0"])
    tets_, u, V = _t(tets).long(), _t(s["u"]), _t(s["V"])
    da, det = _gradients(_t(pos)[tets_])
    w = det.abs()[:, None] * _t(TET_W)
    aw = w @ _t(TET_A)
    Ke = D0 * w.sum(1)[:, None, None] * (da @ da.transpose(1, 2)) + torch.diag_embed(D0 / p["lsf"] ** 2 * aw)
    mag = _t((treg == 1).astype(np.float64))[:, None]
    N = len(pos)

    def nodes(x):
        return torch.zeros(N, x.shape[-1], dtype=F64, device=DEV).index_add_(0, tets_.reshape(-1), x.reshape(-1, x.shape[-1]))

    S = D0 / p["lsd"] ** 2 * nodes((mag * aw)[..., None]) * u
    gV = (V[tets_][:, None] @ da)
    src = mu_e * p["P"] * p["sigma"] * mag[..., None] * w.sum(1)[:, None, None] * (da @ gV.transpose(1, 2)) * u[tets_]
    b = nodes(src)
    fixed, val = torch.zeros(N, 1, dtype=F64, device=DEV), torch.zeros(N, 3, dtype=F64, device=DEV)
    for reg, d in ((0, SPIN_S), (1, [-SPIN_JN * mu_e * x for x in SPIN_UP])):
        at = _t(np.unique(tris[freg == reg])).long()
        fixed[at], val[at] = 1.0, torch.tensor(d, dtype=F64, device=DEV)
    free = 1.0 - fixed

    def K(x):
        # the exchange block of a node: rows (a, S_z, -S_y), (-S_z, a, S_x), (S_y, -S_x, a)
        return nodes(Ke @ x[tets_]) - torch.linalg.cross(S, x)

    D = free / nodes(torch.diagonal(Ke, dim1=1, dim2=2)[..., None])
    x = _bicgstab(lambda y: free * K(y), free * (b - K(val)), torch.zeros_like(b), lambda y: D * y, 1e-13)
    return dict(s=x + val)


def _exact_train(s):
    L = _Llg(s["meshes"])
    u, v = _t(s["u"]), _t(s["v"])
    x, b = L.solve(u, v, _t(s["phi"]), _t(s["phiv"]), _t(s["H"]), s["dt"])
    target = GAMMA0 * x
    feat = torch.cat([u, b / L.mass, v], dim=1)
    e = L.edges
    e = torch.unique(torch.cat([e, e.flip(1)]), dim=0)
    full = torch.cat([feat, torch.zeros_like(u)], dim=1)
    agg = torch.zeros_like(full).index_add_(0, e[:, 0], full[e[:, 1]])
    agg = agg / torch.bincount(e[:, 0], minlength=L.N)[:, None]
    o, n, ns = nv.GUESS_OFFSETS, nv.FG_GUESS_NPARAM, nv.FG_GUESS_NSCALE
    P = _t(s["params"])
    sh, sv, so, sd = (float(a) for a in P[-ns:])
    rounded = P.to(torch.bfloat16).to(F64)  # the forward pass takes the weights in BF16
    P = P.to(F64)
    for a, z in (("W1", "b1"), ("W2", "b2"), ("W3", "b3")):
        P[o[a]:o[z]] = rounded[o[a]:o[z]]
    P = P[:n - ns].requires_grad_(True)

    def part(a, shape):
        return P[o[a]:o[a] + math.prod(shape)].reshape(shape)

    def gelu(z):
        return torch.nn.functional.gelu(z, approximate="tanh")

    sc = torch.tensor([1, 1, 1, sh, sh, sh, sv, sv, sv, sd, sd, sd], dtype=F64, device=DEV)
    z = torch.cat([full * sc, agg * sc], dim=1)
    z = gelu(z @ part("W1", (64, 24)).T + part("b1", (64,)))
    z = gelu(z @ part("W2", (64, 64)).T + part("b2", (64,)))
    w = v + so * (z @ part("W3", (3, 64)).T + part("b3", (3,)))
    norm = 1.0 / (L.N * so * so)
    loss = ((w - _dot(w, u) * u - target) ** 2).sum() * norm
    ref = ((v - _dot(v, u) * u - target) ** 2).sum() * norm
    loss.backward()
    return dict(grad=P.grad, loss=loss.item(), loss_ref=ref.item(), features=feat)


def exact(case, seed):
    c = case
    N, T, F = _sizes(c)
    if c["kind"] in ("run", "field") and (c["steps"] + 1) * N * (5 * T + 4 * F) > 3e11:
        return None  # the exact potentials would take too long
    s = _inputs(c, seed)
    if c["kind"] == "spin":
        return _exact_spin(s)
    if c["kind"] == "train":
        return _exact_train(s)
    return _exact_steps(s)
