"""The work this framework is measured on: implicit cloth steps over the whole
range of sheets (a 13x7 strip to a 512x512 fold), their adjoint, batches of
instances and the standalone broadphase, each through the public entry points
a simulation program calls.

`listed` gives the named cases, `draw` more of the same ranges, `prepare` what
a program holds before the call (a solver initialised on its scene, a state),
`run` one pass (restore the state, advance it, read it back), `work` the bytes
and operations a pass cannot do without, `tolerance` how far another correct
implementation may be off, and `exact` the same pass in plain 64-bit torch
where that is affordable.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

from closim_amd import _abi, scenes
from closim_amd.adjoint import corner_pinned_sheet
from closim_amd.devmem import DeviceArray
from closim_amd.mesh import build_grid, preprocess, sphere_mesh
from closim_amd.scene import (DEFAULT_CONTACT_PARAMS, DEFAULT_MATERIAL, ContactParams, ContactSystem, create_scene)
from closim_amd.solver import HipBatch, HipSolver, _check, load_library

H = scenes.H
NEWTON, PCG = 10, 60  # the solver's default caps


def listed():
    return [
        # an interactive preview: one garment strip of a few dozen vertices, where launches and host reads are all
        dict(name="strip 13x7 fp64", kind="strip", nx=12, ny=6, precision="fp64", precond="jacobi"),
        # a small cloth coming to rest on the floor, default solver: the smallest step with contact
        dict(name="patch 9x9 floor fp64", kind="layers", nx=8, ny=8, layers=1, precision="fp64"),
        # the strip-pull experiment's sheet, reference arithmetic, Jacobi
        dict(name="strip 20x100 fp64", kind="strip", nx=19, ny=99, precision="fp64", precond="jacobi"),
        # the same in mixed precision
        dict(name="strip 20x100 mixed", kind="strip", nx=19, ny=99, precision="mixed", precond="jacobi"),
        # a canopy held in a frame, ordinary resolution, odd sizes, block-Jacobi
        dict(name="canopy 131x90 mixed", kind="canopy", nx=130, ny=89, precision="mixed", precond="block"),
        # two layers lying on each other above the floor, friction: self contact in numbers
        dict(name="layers 2x33x33 fp64", kind="layers", nx=32, ny=32, layers=2, precision="fp64"),
        # the sphere + floor drape at the moment of contact, both precisions
        dict(name="drape 256x256 fp64", kind="drape", nx=255, precision="fp64"),
        dict(name="drape 256x256 mixed", kind="drape", nx=255, precision="mixed"),
        # the self-contact fold with additive Schwarz, the largest step, both precisions
        dict(name="fold 512x512 fp64", kind="fold", nx=511, precision="fp64", target=64),
        dict(name="fold 512x512 mixed", kind="fold", nx=511, precision="mixed", target=64),
        # a dozen uneven drapes advanced together, as a training or fitting loop does
        dict(name="batch of 12 drapes mixed", kind="batch", count=12, meshes=0xB47C4),
        # backward: the adjoint of one step of the material-fitting sheet
        dict(name="adjoint 128x128", kind="adjoint", nx=127),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["strip", "canopy", "layers", "drape", "fold", "batch", "adjoint", "pairs"])
    prec = rng.choice(["fp64", "mixed"])
    if kind == "strip":
        return dict(kind=kind, nx=log(4, 60), ny=log(5, 160), precision=prec, precond="jacobi")
    if kind == "canopy":
        return dict(kind=kind, nx=log(20, 160), ny=log(20, 160), precision=prec, precond=rng.choice(["jacobi", "block"]))
    if kind == "layers":
        return dict(kind=kind, nx=log(6, 48), ny=log(6, 48), layers=rng.choice([1, 2, 3]), precision="fp64")
    if kind == "drape":
        return dict(kind=kind, nx=log(30, 255), precision=prec)
    if kind == "fold":
        return dict(kind=kind, nx=log(40, 500), precision=prec, target=rng.choice([16, 32, 64]))
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(2, 12), meshes=rng.randrange(1, 1 << 20))
    if kind == "adjoint":
        return dict(kind=kind, nx=log(16, 127))
    return dict(kind=kind, nx=log(40, 511), ny=log(40, 511))


# ---- scenes -----------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _sheet(nx, ny, w, h, density, layers=1, gap=0.0):
    """`layers` flat sheets of one size above each other, preprocessed."""
    g = [build_grid(nx, ny, w, h) for _ in range(layers)]
    P = [p.reshape(-1, 3).copy() for p, _, _ in g]
    for k in range(layers):
        P[k][:, 1] = k * gap
    return preprocess(*scenes.merge_parts([(p.reshape(-1), uv, idx) for p, (_, uv, idx) in zip(P, g)]), density)


def _waves(rng, X, count, lo, hi):
    """A smooth random field over the rest positions, of values within +-1."""
    out = np.zeros(len(X))
    a = rng.uniform(0.5, 1.5, count)
    for k in range(count):
        kx, kz = rng.uniform(lo, hi, 2) * rng.choice([-1, 1], 2)
        out += a[k] / a.sum() * np.sin(kx * X[:, 0] + kz * X[:, 2] + rng.uniform(0, 2 * math.pi))
    return out


def _contact(d_hat, mu):
    return ContactSystem(ContactParams(dHatM=d_hat, kappaJ=50.0, dMinM=1e-4, frictionMu=mu, frictionEpsM=1e-4))


def _scene(case, seed):
    """The scene with the state a program holds before the step."""
    rng = np.random.default_rng(int(seed))
    kind = case["kind"]
    mat = scenes.STRIP_MATERIAL
    if kind in ("strip", "canopy"):
        # hung vertically, 1 cm per cell, taut and swinging out of its plane: the pulled strip held by its top and
        # bottom rows, the canopy by its whole border
        nx, ny = case["nx"], case["ny"]
        mesh = _sheet(nx, ny, 0.01 * nx, 0.01 * ny, mat.arealDensityKgM2)
        sc = create_scene(mesh, mat)
        X = sc.positions.reshape(-1, 3)
        rest = X.copy()
        wide = rng.uniform(0.01, 0.03) if kind == "canopy" else 0.002
        X[:, 0] = rest[:, 0] * (1 + wide) + 1e-5 * _waves(rng, rest, 4, 5, 25)
        X[:, 1] = -rest[:, 2] * (1 + rng.uniform(0.01, 0.03)) + 1e-5 * _waves(rng, rest, 4, 5, 25)
        X[:, 2] = 0.001 * _waves(rng, rest, 4, 5, 25)
        sc.velocities.reshape(-1, 3)[:, 2] = 0.05 * _waves(rng, rest, 4, 3, 12)
        i = np.arange(mesh.count)
        held = (i <= nx) | (i >= ny * (nx + 1))
        if kind == "canopy":
            held |= (i % (nx + 1) == 0) | (i % (nx + 1) == nx)
        for j in i[held]:
            sc.pinned[int(j)] = tuple(float(c) for c in X[j])
        return sc
    if kind == "layers":
        # sheets of 4 mm cells, 1.3 mm apart and above the floor (d_hat 2 mm), sinking
        nx, ny = case["nx"], case["ny"]
        mesh = _sheet(nx, ny, 0.004 * nx, 0.004 * ny, 0.15, case["layers"], 0.0013)
        sc = create_scene(mesh, DEFAULT_MATERIAL)
        X = sc.positions.reshape(-1, 3)
        X[:, 1] += 0.0013
        X += rng.uniform(-1e-4, 1e-4, X.shape)
        sc.velocities.reshape(-1, 3)[:, 1] = -0.02 + 0.02 * _waves(rng, X, 3, 10, 60)
        sc.contact = ContactSystem(DEFAULT_CONTACT_PARAMS)
        sc.contact.setFloor(0.0)
        return sc
    if kind == "drape":
        # the sheet of the sphere drape as it reaches the sphere's top
        nx = case["nx"]
        mesh = _sheet(nx, nx, 1.0, 1.0, mat.arealDensityKgM2)
        sc = create_scene(mesh, mat)
        X = sc.positions.reshape(-1, 3)
        X[:, 1] = 0.45 + rng.uniform(6e-4, 9e-4)
        X += rng.uniform(-1e-4, 1e-4, X.shape)
        sc.velocities.reshape(-1, 3)[:, 1] = rng.uniform(-0.3, -0.1) + 0.05 * _waves(rng, X, 4, 4, 16)
        sc.contact = _contact(1e-3, 0.3)
        sc.contact.setFloor(0.0)
        sc.contact.setStaticMesh(*sphere_mesh(0.25, 64, 32, center=(0.5, 0.2, 0.5)))
        return sc
    if kind == "fold":
        # the crumpled sheet of the fold as its valleys reach the floor, at the same density of vertices
        nx = case["nx"]
        side = 1.5 * nx / 511
        mesh = _sheet(nx, nx, side, side, mat.arealDensityKgM2)
        sc = create_scene(mesh, mat)
        X = sc.positions.reshape(-1, 3)
        X[:, 1] = 0.05 * _waves(rng, X, int(rng.integers(3, 7)), 4, 24)
        X[:, 1] += rng.uniform(4e-4, 1e-3) - X[:, 1].min()
        sc.velocities.reshape(-1, 3)[:, 1] = rng.uniform(-0.5, -0.1)
        sc.contact = _contact(5e-4, 0.4)
        sc.contact.setFloor(0.0)
        return sc
    # adjoint: the corner-pinned sheet under light tension, with shallow waves
    sc = corner_pinned_sheet(case["nx"])
    X = sc.positions.reshape(-1, 3)
    rest = X.copy()
    X[:, [0, 2]] *= 1 + rng.uniform(0.002, 0.004, 2)
    X[:, 1] += 0.004 * _waves(rng, rest, 4, 3, 10)
    for i in sc.pinned:
        sc.pinned[i] = tuple(float(c) for c in X[i])
    sc.velocities.reshape(-1, 3)[:] = 0.05 * rng.standard_normal(3)
    return sc


def _options(case):
    pre = {"jacobi": _abi.CS_PRECOND_JACOBI, "block": _abi.CS_PRECOND_BLOCK_JACOBI}
    if case["kind"] in ("strip", "canopy"):
        return dict(precond=pre[case["precond"]])
    if case["kind"] == "drape":
        return dict(precond=pre["block"], flags=_abi.CS_FLAG_DEVICE_NEWTON)
    if case["kind"] == "fold":
        t = case["target"]
        return dict(precond=_abi.CS_PRECOND_SCHWARZ, schwarz=(t, 1, t),
                    flags=_abi.CS_FLAG_DEVICE_NEWTON | _abi.CS_FLAG_BREAKDOWN_DESCENT)
    if case["kind"] == "batch":
        return dict(precond=pre["block"], flags=_abi.CS_FLAG_DEVICE_NEWTON)
    return {}


@functools.lru_cache(maxsize=None)
def _batch_scenes(count, meshes):
    return scenes.batch_drapes(count, meshes)


def _adjoint_inputs(case, seed):
    """x_prev, v_prev, x_next and the loss's gradients of one step."""
    sc = _scene(case, seed)
    rng = np.random.default_rng([int(seed), 1])
    x1 = sc.positions.copy()
    v0 = sc.velocities.copy()
    x0 = x1 - H * v0
    n3 = len(x1)
    return sc, x0, v0, x1, rng.standard_normal(n3) / n3, 0.01 * rng.standard_normal(n3) / n3


# ---- one pass ---------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "pairs":
        # a fold's triangles swept over one step, device arrays and a pair buffer of the size such a program keeps
        nx, ny = case["nx"], case["ny"]
        rng = np.random.default_rng(int(seed))
        mesh = _sheet(nx, ny, 0.003 * nx, 0.003 * ny, 0.2)
        X = mesh.positions.astype(np.float64).reshape(-1, 3).copy()
        X[:, 1] = 0.05 * _waves(rng, X, 4, 4, 24)
        Y = X + rng.uniform(-1e-3, 1e-3, 3) + rng.uniform(-1e-4, 1e-4, X.shape)
        cap = 16 * mesh.tri_count
        return dict(kind=kind, x0=DeviceArray(X.reshape(-1)), x1=DeviceArray(Y.reshape(-1)),
                    idx=DeviceArray(mesh.indices), n=mesh.count, m=mesh.tri_count, cap=cap,
                    out=DeviceArray(dtype=np.uint32, shape=(cap, 2)))
    if kind == "batch":
        # each sheet of the batch just above its sphere
        rng = np.random.default_rng(int(seed))
        solvers, states = [], []
        for sc in _batch_scenes(case["count"], case["meshes"]):
            x, v = sc.mesh.positions.astype(np.float64), np.zeros_like(sc.velocities)
            x.reshape(-1, 3)[:, 1] = 0.45 + rng.uniform(6e-4, 9e-4)
            x += rng.uniform(-1e-4, 1e-4, x.shape)
            v.reshape(-1, 3)[:, 1] = rng.uniform(-0.3, -0.1)
            own = create_scene(sc.mesh, sc.material, sc.gravity)
            own.contact = sc.contact
            g = HipSolver("mixed", **_options(case))
            g.initialize(own)
            solvers.append(g)
            states.append((x, v))
        return dict(kind=kind, batch=HipBatch(solvers, packed=True), solvers=solvers, states=states)
    if kind == "adjoint":
        sc, *inputs = _adjoint_inputs(case, seed)
        g = HipSolver("fp64", **_options(case))
        g.initialize(sc)
        return dict(kind=kind, g=g, inputs=inputs)
    sc = _scene(case, seed)
    x, v = sc.positions.copy(), sc.velocities.copy()
    g = HipSolver(case["precision"], **_options(case))
    g.initialize(sc)
    return dict(kind="step", g=g, x=x, v=v)


def run(state):
    kind = state["kind"]
    if kind == "step":
        g = state["g"]
        g.set_state(state["x"], state["v"])
        g.step(H)
        return g.getPositions(), g.getVelocities()
    if kind == "batch":
        for g, (x, v) in zip(state["solvers"], state["states"]):
            g.set_state(x, v)
        state["batch"].step(H)
        return [(g.getPositions(), g.getVelocities()) for g in state["solvers"]]
    if kind == "adjoint":
        dx, dv, dtheta, _, _ = state["g"].step_adjoint(H, *state["inputs"])
        return dx, dv, dtheta
    cnt = C.c_uint64()
    _check(load_library().cs_broadphase_self_pairs(0, state["x0"].ptr, state["x1"].ptr, state["n"], state["idx"].ptr,
                                                   state["m"], 5e-4, state["out"].ptr, state["cap"], C.byref(cnt),
                                                   None, None))
    return state["out"].numpy(cnt.value)


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    """Bytes and operations: the mesh and the state read and written once for
    every gradient, energy and Hessian product of the capped Newton and PCG
    iterations (40n + 32m bytes of an FP32 product, 80n + 52m in FP64; about
    200 operations a triangle and product, 24 dihedrals of 60 a hinge and
    gradient), and the Schwarz factor's tiles once per apply."""
    kind = case["kind"]
    if kind == "pairs":
        m = 2.0 * case["nx"] * case["ny"]
        return {"bytes": 12 * m + 24 * m + 8 * 2.5 * m, "flops": 60 * m}
    if kind == "batch":
        n = sum(sc.mesh.count for sc in _batch_scenes(case["count"], case["meshes"]))
    elif kind == "layers":
        n = case["layers"] * (case["nx"] + 1) * (case["ny"] + 1)
    else:
        n = (case["nx"] + 1) * (case.get("ny", case["nx"]) + 1)
    m, hinges = 2.0 * n, 3.0 * n
    if kind == "adjoint":
        its = 15.0 * case["nx"]  # block-Jacobi PCG to 1e-10 grows with the sheet's width in cells
        return {"bytes": its * (80 * n + 52 * m + 72 * hinges) + 13 * 24 * n,
                "flops": its * (200 * m + 1000 * hinges)}
    fp64 = case.get("precision", "mixed") == "fp64"
    pcg = {"strip": 35, "canopy": 15, "layers": 30, "drape": 20, "fold": 9, "batch": 25}[kind]
    hvp = 80 * n + 52 * m if fp64 else 40 * n + 32 * m
    newton = 96 * n + 32 * m + 40 * hinges
    factor = {"fold": (8 if fp64 else 4) * 3 * n * (3 * case.get("target", 0) + 1) / 2}.get(kind, 0.0)
    return {"bytes": 96 * n + NEWTON * (pcg * (hvp + factor) + 3 * newton),
            "flops": NEWTON * (pcg * 200 * m + 2 * 100 * m + 26 * 60 * hinges)}


def tolerance(case):
    if case["kind"] == "pairs":
        return "exact"
    if case["kind"] == "adjoint":
        return {"rel": 1e-6}  # PCG to 1e-10; kb's gradient differences energies (3e-7 off exact)
    # A step stops at its caps, far from the root, and its PCG where curvature turns negative: summing left to right
    # instead of with correct rounding moves the velocities of these states by 1e-4 to 1e-2 in 64 bits already.
    return {"rel": 0.03}


# ---- the same in plain 64-bit torch -----------------------------------------

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


class _Exact:
    """Energies, gradients and Hessian products of a contact-free scene."""

    def __init__(self, sc):
        d = _dev()
        self.d, self.sc = d, sc
        me, mat = sc.mesh, sc.material
        self.n = me.count
        self.tri = torch.from_numpy(me.indices.astype(np.int64)).to(d).view(-1, 3)
        self.inv = torch.from_numpy(me.inv_dm.astype(np.float64)).to(d).view(-1, 2, 2)  # [[a, b], [c, d]]
        self.area = torch.from_numpy(me.areas.astype(np.float64)).to(d)
        self.mass = torch.from_numpy(me.masses.astype(np.float64)).to(d)
        self.hv = torch.from_numpy(me.hinge_verts.astype(np.int64)).to(d)
        self.rest, self.w = (torch.from_numpy(np.asarray(a, np.float64)).to(d) for a in
                             (me.hinge_rest, me.hinge_len ** 2 / np.maximum(me.hinge_area, 1e-12)))
        self.mod = (mat.stretchWarp, mat.stretchWeft, mat.stretchCoupling, mat.shear)
        self.kb, self.thick = 0.5 * (mat.bendWarp + mat.bendWeft), mat.thickness
        self.free = torch.ones(self.n, 1, dtype=torch.float64, device=d)
        self.pins = torch.tensor(sorted(sc.pinned), dtype=torch.int64, device=d)
        self.pin_pos = torch.tensor([sc.pinned[i] for i in sorted(sc.pinned)], dtype=torch.float64, device=d).view(-1, 3)
        self.free[self.pins] = 0

    def pin(self, x):
        x = x.clone()
        x[self.pins] = self.pin_pos
        return x

    def deform(self, x):  # (m, 3, 2): e1 a + e2 c, e1 b + e2 d
        t = x[self.tri]
        return torch.stack([t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]], 2) @ self.inv

    def stress(self, E, mod):
        c00, c11, c01, g = mod
        s00, s11, s01 = c00 * E[:, 0, 0] + c01 * E[:, 1, 1], c11 * E[:, 1, 1] + c01 * E[:, 0, 0], 2 * g * E[:, 0, 1]
        return torch.stack([s00, s01, s01, s11], 1).view(-1, 2, 2)

    def scatter(self, P):
        G = (self.thick * self.area)[:, None, None] * (P @ self.inv.transpose(1, 2))
        out = torch.zeros(self.n, 3, dtype=torch.float64, device=self.d)
        for c, g in enumerate((-(G[:, :, 0] + G[:, :, 1]), G[:, :, 0], G[:, :, 1])):
            out.index_add_(0, self.tri[:, c], g)
        return out

    def membrane(self, x, mod):
        F = self.deform(x)
        E = 0.5 * (F.transpose(1, 2) @ F - torch.eye(2, dtype=torch.float64, device=self.d))
        return F, E, self.stress(E, mod)

    def bend(self, x, k):
        p = x[self.hv]
        e, a, b = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0], p[:, 3] - p[:, 0]
        n1, n2 = torch.linalg.cross(e, a), torch.linalg.cross(e, b)
        # the unsigned angle between the normals, well conditioned where they are (anti)parallel
        s = torch.linalg.cross(n1, n2).square().sum(1)
        th = torch.atan2(torch.sqrt(s + 1e-300), (n1 * n2).sum(1))
        return (0.5 * k * (th - self.rest) ** 2 * self.w).sum()

    def bend_grad(self, x, k, graph=False):
        y = x.detach().clone().requires_grad_(True)
        g, = torch.autograd.grad(self.bend(y, k), y, create_graph=graph)
        return (g, y) if graph else g

    def energy(self, x, yhat):
        _, E, S = self.membrane(x, self.mod)
        c00, c11, c01, g = self.mod
        psi = (0.5 * c00 * E[:, 0, 0] ** 2 + 0.5 * c11 * E[:, 1, 1] ** 2 + c01 * E[:, 0, 0] * E[:, 1, 1] +
               2 * g * E[:, 0, 1] ** 2)
        inertia = (0.5 * self.mass[:, None] * (x - yhat) ** 2 / (H * H)).sum()
        return float(inertia + (self.thick * self.area * psi).sum() + self.bend(x, self.kb))

    def grad(self, x, yhat):
        F, _, S = self.membrane(x, self.mod)
        g = self.mass[:, None] * (x - yhat) / (H * H) + self.scatter(F @ S) + self.bend_grad(x, self.kb)
        return g * self.free

    def hvp(self, FS, p):
        F, S = FS
        dF = self.deform(p)
        FdF = F.transpose(1, 2) @ dF
        dS = self.stress(0.5 * (FdF + FdF.transpose(1, 2)), self.mod)
        return (self.mass[:, None] / (H * H) * p + self.scatter(dF @ S + F @ dS)) * self.free

    def blocks(self, FS, diag):
        """3x3 vertex blocks of the membrane Hessian plus the diagonal, inverted."""
        F, S = FS
        B = torch.zeros(self.n, 3, 3, dtype=torch.float64, device=self.d)
        K = torch.stack([-(self.inv[:, 0] + self.inv[:, 1]), self.inv[:, 0], self.inv[:, 1]], 1)
        for c in range(3):
            k = K[:, c]
            for i in range(3):
                dF = torch.zeros_like(F)
                dF[:, i] = k
                FdF = F.transpose(1, 2) @ dF
                dP = dF @ S + F @ self.stress(0.5 * (FdF + FdF.transpose(1, 2)), self.mod)
                B[:, :, i].index_add_(0, self.tri[:, c], (self.thick * self.area)[:, None] * (dP @ k[:, :, None])[:, :, 0])
        B = 0.5 * (B + B.transpose(1, 2)) + diag[:, None, None] * torch.eye(3, dtype=torch.float64, device=self.d)
        ok = (torch.linalg.eigvalsh(B) > 0).all(1)
        B[~ok] = diag[~ok][:, None, None] * torch.eye(3, dtype=torch.float64, device=self.d)
        return torch.linalg.inv(B)


def _exact_step(case, sc):
    """The step's algorithm: predictor, Newton with truncated PCG (relative
    tolerance 1e-3), steepest descent where that is no descent direction, a
    trust region of 2 mm, Armijo halving."""
    X = _Exact(sc)
    mat = sc.material
    x0 = torch.from_numpy(sc.positions).to(X.d).view(-1, 3)
    v0 = torch.from_numpy(sc.velocities).to(X.d).view(-1, 3)
    yhat = x0 + H * v0 + H * H * torch.tensor(sc.gravity, dtype=torch.float64, device=X.d)
    x = X.pin(yhat)
    E = X.energy(x, yhat)
    beta = max(mat.stretchWarp, mat.stretchWeft, mat.shear) * mat.thickness * 0.1 + 1e-6
    diag = X.mass / (H * H) + beta
    for _ in range(NEWTON):
        g = X.grad(x, yhat)
        if float(g.norm()) < 1e-5:
            break
        F, _, S = X.membrane(x, X.mod)
        if case["precond"] == "block":
            B = X.blocks((F, S), diag)
            pre = lambda r: (B @ r[:, :, None])[:, :, 0] * X.free  # noqa: E731
        else:
            pre = lambda r: r / diag[:, None] * X.free  # noqa: E731
        dx, r = torch.zeros_like(g), -g
        z = pre(r)
        p, rz = z, float((r * z).sum())
        tol = max(1e-3 * max(float(g.norm()), 1e-12), 1e-12)
        for _ in range(PCG):
            Ap = X.hvp((F, S), p)
            pAp = float((p * Ap).sum())
            if not pAp > 1e-30:
                break
            a = rz / pAp
            dx, r = dx + a * p, r - a * Ap
            if float(r.norm()) < tol:
                break
            z = pre(r)
            rz, old = float((r * z).sum()), rz
            p = z + rz / old * p
        gd = float((g * dx).sum())
        if not gd < 0:
            dx = -g / diag[:, None]
            gd = float((g * dx).sum())
        top = float(dx.abs().max())
        if top > 0.002:
            dx, gd = dx * (0.002 / top), gd * (0.002 / top)
        alpha, ok = 1.0, False
        for _ in range(10):
            xt = X.pin(x + alpha * dx)
            Et = X.energy(xt, yhat)
            if Et <= E + 1e-4 * alpha * gd:
                x, E, ok = xt, Et, True
                break
            alpha *= 0.5
        if not ok or alpha < 1e-6:
            break
    v = (x - x0) / H * (1 - min(max(mat.damping, 0), 0.1))
    return x.reshape(-1).cpu().numpy(), v.reshape(-1).cpu().numpy()


def _exact_adjoint(case, seed):
    """H lambda = dL/dx1 + (damp / h) dL/dv1 on the free vertices by CG, then
    the products with the step's derivatives."""
    sc, x0, v0, x1, gx, gv = _adjoint_inputs(case, seed)
    X = _Exact(sc)
    mat = sc.material
    gx, gv, x = (torch.from_numpy(a).to(X.d).view(-1, 3) for a in (gx, gv, x1))
    damp = 1 - min(max(mat.damping, 0), 0.1)
    F, _, S = X.membrane(x, X.mod)
    gb, y = X.bend_grad(x, X.kb, graph=True)

    def A(p):
        return (X.hvp((F, S), p) + torch.autograd.grad((gb * p).sum(), y, retain_graph=True)[0]) * X.free

    B = X.blocks((F, S), X.mass / (H * H))
    r = (gx + damp / H * gv) * X.free
    lam, z = torch.zeros_like(r), (B @ r[:, :, None])[:, :, 0] * X.free
    p, rz, stop = z, (r * z).sum(), 1e-13 * float(r.norm())
    for k in range(20 * case["nx"] + 400):
        Ap = A(p)
        a = rz / (p * Ap).sum()
        lam, r = lam + a * p, r - a * Ap
        if k % 16 == 0 and float(r.norm()) < stop:
            break
        z = (B @ r[:, :, None])[:, :, 0] * X.free
        rz, old = (r * z).sum(), rz
        p = z + rz / old * p
    dth = []
    for j in range(4):
        F, _, S = X.membrane(x, tuple(float(i == j) for i in range(4)))
        dth.append(-float((lam * X.scatter(F @ S)).sum()))
    dth.append(-float((lam * X.bend_grad(x, 1.0)).sum()))
    dx = lam * X.mass[:, None] / (H * H) - damp / H * gv
    dv = lam * X.mass[:, None] / H
    return dx.reshape(-1).cpu().numpy(), dv.reshape(-1).cpu().numpy(), np.array(dth)


def exact(case, seed):
    if case["kind"] in ("strip", "canopy"):
        # the velocities of a truncated solve hold its round-off divided by the time step (see tolerance)
        return _exact_step(case, _scene(case, seed))[0], None
    if case["kind"] == "adjoint":
        return _exact_adjoint(case, seed)
    # pairs: whole numbers, nothing to round.  The contact steps in plain torch (all candidate primitives, their
    # times of impact and the line search over them, thousands of kernels per iteration) take minutes.
    return None
