"""Performance cases of the PDLSM-FEM library: the calls a user's program makes, over the sizes it makes them at.

A case is a dict of plain values with a "kind":

  explicit   explicit central difference (`Context.explicit_run`): lumped or consistent mass, FP64 or FP32 force
  static     assembly and static solve of one load case (`assemble`, `static_solve`)
  newmark    implicit Newmark steps (`newmark_run`)
  loadstep   the device part of a quasi-static load step: K and the residual force, then the nodal stresses
  csr        K and F in the reference's CSR layout on the host, and the PARDISO seam on them (`solve_csr`)
  learned    training gradient, BF16 smoother prediction and the learned solve of a cracked plate
  families   the per-node families of a node cloud (`FamilyBatch`)

Meshes are the generators of workloads.py (plates, boxes, cracked plates, penny-cracked boxes), the ones the
tests and the benchmark use.  exact() restates the whole path in plain torch, FP64: element by element and bond by
bond, without the library.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pdlsm-fem_mpi_amd")


def _load(name, file, **kw):
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, os.path.join(_PKG, file), **kw)
        sys.modules[name] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[name])
    return sys.modules[name]


def _pdx():
    return _load("pdlsm_fem_mpi_amd", "__init__.py", submodule_search_locations=[_PKG])


def _workloads():
    return _load("pdlsm_fem_mpi_amd_workloads", "workloads.py")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a small plate stepped a few times between two results: the call itself counts
        dict(name="explicit-plate", kind="explicit", mesh="plate", nx=61, ny=31, lumped=True, fp32=False, steps=12),
        # the benchmark's box, a few hundred steps between two result files, in both force precisions
        dict(name="explicit-box60", kind="explicit", mesh="box", n=60, pd=20, lumped=True, fp32=False, steps=300),
        dict(name="explicit-box60-fp32", kind="explicit", mesh="box", n=60, pd=20, lumped=True, fp32=True, steps=300),
        # consistent mass, the command files' default: a mass solve in every step
        dict(name="explicit-box31-consistent", kind="explicit", mesh="box", n=31, pd=10, lumped=False, fp32=False, steps=10),
        # one load case of the cracked plate and of a box: assembly, coarse space, solve to 1e-8
        dict(name="static-crack501", kind="static", mesh="crack", nx=501, ny=251, fp32=False),
        dict(name="static-box41-fp32", kind="static", mesh="box", n=41, pd=13, fp32=True),
        # implicit steps at ten times the critical step: the penny-cracked box, and a small cracked plate
        dict(name="newmark-penny80-fp32", kind="newmark", mesh="penny", n=80, pd=24, fp32=True, mirrored=True, steps=4),
        dict(name="newmark-plate", kind="newmark", mesh="crack", nx=121, ny=61, fp32=False, mirrored=False, steps=6),
        # one load step's assembly, residual force and stress recovery on the benchmark's box
        dict(name="loadstep-box60", kind="loadstep", mesh="box", n=60, pd=20),
        # the drop-in seam: K and F handed over in CSR and solved there
        dict(name="csr-plate", kind="csr", mesh="plate", nx=201, ny=101),
        # one training gradient, one prediction and one solve with the learned smoother
        dict(name="learned-crack251", kind="learned", mesh="crack", nx=251, ny=126, probes=8),
        # a node cloud whose families come back whole
        dict(name="families-20", kind="families", n=20),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["explicit", "explicit", "explicit", "static", "newmark", "newmark", "loadstep", "csr", "learned",
                       "families"])
    if kind == "explicit":
        fp32 = rng.random() < 0.5
        if rng.random() < 0.3:
            nx = _log(rng, 31, 301)
            return dict(kind=kind, mesh="plate", nx=nx, ny=max(15, int(nx * rng.uniform(0.4, 0.8))),
                        lumped=rng.random() < 0.7, fp32=fp32, steps=_log(rng, 6, 60))
        lumped = rng.random() < 0.7
        n = _log(rng, 12, 60) if lumped else _log(rng, 12, 40)
        return dict(kind=kind, mesh="box", n=n, pd=max(4, int(n * rng.uniform(0.2, 0.4))), lumped=lumped, fp32=fp32,
                    steps=_log(rng, 6, 300) if lumped else _log(rng, 4, 16))
    if kind == "static":
        if rng.random() < 0.5:
            nx = _log(rng, 81, 501)
            return dict(kind=kind, mesh="crack", nx=nx, ny=nx // 2 + rng.randrange(1, 9), fp32=rng.random() < 0.5)
        n = _log(rng, 14, 41)
        return dict(kind=kind, mesh="box", n=n, pd=max(4, n // 3), fp32=rng.random() < 0.5)
    if kind == "newmark":
        fp32, mirrored = rng.random() < 0.5, rng.random() < 0.5
        if rng.random() < 0.4:
            nx = _log(rng, 61, 301)
            return dict(kind=kind, mesh="crack", nx=nx, ny=nx // 2 + rng.randrange(1, 9), fp32=False, mirrored=mirrored,
                        steps=rng.randrange(3, 8))
        n = _log(rng, 20, 72)
        return dict(kind=kind, mesh="penny", n=n, pd=max(4, int(n * 0.3)), fp32=fp32, mirrored=mirrored,
                    steps=rng.randrange(2, 5))
    if kind == "loadstep":
        if rng.random() < 0.3:
            nx = _log(rng, 61, 501)
            return dict(kind=kind, mesh="crack", nx=nx, ny=nx // 2 + rng.randrange(1, 9))
        n = _log(rng, 12, 60)
        return dict(kind=kind, mesh="box", n=n, pd=max(4, int(n * rng.uniform(0.2, 0.4))))
    if kind == "csr":
        nx = _log(rng, 41, 201)
        return dict(kind=kind, mesh="plate", nx=nx, ny=max(15, int(nx * rng.uniform(0.4, 0.6))))
    if kind == "learned":
        nx = _log(rng, 81, 301)
        return dict(kind=kind, mesh="crack", nx=nx, ny=nx // 2 + rng.randrange(1, 9), probes=rng.randrange(2, 9))
    return dict(kind=kind, n=rng.randrange(9, 21))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _mesh(case, seed):
    """The case's mesh and loads, from the seed alone."""
    W = _workloads()
    rng = np.random.default_rng(seed + 1)
    load = rng.uniform(0.5, 2.0)
    if case["mesh"] == "plate":
        nx, ny, dx = case["nx"], case["ny"], 5e-4
        width = (nx - 1) * dx
        mesh = W.plate2d(nx=nx, ny=ny, dx=dx, pd_x=(0.4 * width, 0.6 * width), ux_right=1e-5 * load)
        # interior nodes off the grid, as a meshed part has them; the pattern of K follows the mesh, so where K comes
        # back the mesh is one for all seeds and the material differs
        shape = np.random.default_rng(nx * ny) if case["kind"] == "csr" else rng
        i, j = np.arange(nx * ny) % nx, np.arange(nx * ny) // nx
        inner = (i > 0) & (i < nx - 1) & (j > 0) & (j < ny - 1)
        mesh["x"][inner, :2] += shape.uniform(-0.1, 0.1, (int(inner.sum()), 2)) * dx
        if case["kind"] == "csr":
            mesh["E"] *= rng.uniform(0.5, 1.5)
            mesh["nu"] = rng.uniform(0.2, 0.35)
        # a traction on the upper edge besides the prescribed displacement
        a = np.arange(1, nx) + (ny - 1) * nx
        mesh["nbc"] = [dict(con=np.stack([a + 1, a], 1).astype(np.int32), val=1e6 * load)]
    elif case["mesh"] == "box":
        mesh = W.box3d(n=case["n"], pd_block=case["pd"], seed=seed, traction=1e6 * load)
        dx = 1e-3
    elif case["mesh"] == "crack":
        dx = 2e-4
        mesh = W.crack2d(seed=seed, nx=case["nx"], ny=case["ny"], dx=dx, uy_top=1e-5 * load)
    else:
        dx = 1e-3
        mesh = W.penny3d(n=case["n"], dx=dx, pd_block=case["pd"], t_final=5e6 * load)
    mesh["lumped_mass"] = bool(case.get("lumped", True))
    # wave speed of the material: the critical step is about dx / c for a lumped mass and regular elements
    c = math.sqrt(mesh["E"] / mesh["rho"] * (1 - mesh["nu"]) / ((1 + mesh["nu"]) * (1 - 2 * mesh["nu"])))
    mesh["dt"] = (10.0 if case["kind"] == "newmark" else 0.25 if mesh["lumped_mass"] else 0.12) * dx / c
    if case["kind"] == "newmark":
        if case["mesh"] == "penny":
            mesh["nbc"][0]["vel"] = 5e6 * load / (50 * mesh["dt"])
        else:
            # the plate's upper edge is pulled at a constant rate
            mesh["ebc"][2].update(val=0.0, vel=1e-6 * load / mesh["dt"], vary=True)
    return mesh


def _field(mesh, seed):
    """A smooth displacement field with a little noise, zero strain nowhere."""
    rng = np.random.default_rng(seed + 2)
    x, d = np.asarray(mesh["x"]), mesh["dim"]
    s = x[:, :d] / x[:, :d].max()
    u = 1e-4 * x[:, :d].max() * (np.sin(s @ rng.uniform(-3, 3, (d, d))) + s @ rng.uniform(-1, 1, (d, d)))
    return np.ascontiguousarray(u + 1e-9 * rng.standard_normal(u.shape)).ravel()


def _cloud(case, seed):
    """A node cloud whose families are the same for all seeds, with the seed's node volumes and material."""
    c = _workloads().family_batch(n=case["n"], seed=case["n"])
    rng = np.random.default_rng(seed + 4)
    c["vol"] = c["vol"] * rng.uniform(0.7, 1.3, len(c["vol"]))
    E, nu = 70e9 * rng.uniform(0.5, 1.5), rng.uniform(0.2, 0.35)
    return c, E * nu / ((1 - 2 * nu) * (1 + nu)), 0.5 * E / (1 + nu)


_NLF = 0.33


def prepare(case, seed):
    pdx, kind = _pdx(), case["kind"]
    if kind == "families":
        c, lam, mu = _cloud(case, seed)
        fb = pdx.FamilyBatch(c["x"], c["vol"], c["delta"], nlf=_NLF, lam=lam, mu=mu, dim=3)
        return dict(case=case, fb=fb, off=fb.families()[0])
    mesh = _mesh(case, seed)
    model = pdx.Model(mesh)
    s = dict(case=case, model=model, cx=pdx.Context(model, 0))
    if kind == "loadstep":
        s["u"] = _field(mesh, seed)
        s["cx"].set_dof_values(s["u"])
    if kind == "csr":
        s["ia"], s["ja"] = model.csr()
    if kind == "learned":
        s["gnn"] = pdx.GNN(2, 0, seed=seed % 1000003)
        # the untrained network has a zero head: give every weight a value, so that the smoother is not block Jacobi
        w = s["gnn"].params()
        w += np.random.default_rng(seed + 3).uniform(-0.02, 0.02, w.size).astype(np.float32)
        s["gnn"].set_params(w)
        s["cx"].assemble(pdx.PDX_MODE_STATIC, want_K=False)
        s["probe_seed"] = seed % 1000003
    return s


def run(s):
    pdx, case = _pdx(), s["case"]
    kind = case["kind"]
    prec = pdx.PDX_FP32 if case.get("fp32") else pdx.PDX_FP64
    if kind == "families":
        s["fb"].run()
        A, L, H = s["fb"].results(0, s["fb"].n_fam, s["off"])
        return dict(A=A, L=L, H=H)
    cx = s["cx"]
    if kind == "explicit":
        u, up = cx.explicit_run(case["steps"], prec)
        return dict(u=u, u_prev=up)
    if kind == "static":
        _, F = cx.assemble(pdx.PDX_MODE_STATIC, want_K=False)
        u, _ = cx.static_solve(pdx.solve_opts(precond=pdx.PDX_PREC_TWO_LEVEL, precision=prec, tol=1e-8))
        return dict(F=F, u=u)
    if kind == "newmark":
        o = pdx.solve_opts(precond=pdx.PDX_PREC_BLOCK_JACOBI, precision=prec, tol=1e-8, mirrored=case["mirrored"])
        u, v, a, _ = cx.newmark_run(case["steps"], o)
        return dict(u=u, v=v, a=a)
    if kind == "loadstep":
        _, F = cx.assemble(pdx.PDX_MODE_QUASI, want_K=False)
        return dict(F=F, sigma=cx.node_stresses(s["u"]))
    if kind == "csr":
        K, F = cx.assemble(pdx.PDX_MODE_STATIC)
        # it stands in for a direct solver, so the tolerance is tighter
        x, _ = pdx.solve_csr(s["ia"], s["ja"], K, F, pdx.solve_opts(tol=1e-10))
        return dict(K=K, F=F, x=x)
    loss, grad = s["gnn"].loss_grad(cx, n_probes=case["probes"], probe_seed=s["probe_seed"])
    M, _ = s["gnn"].infer(cx, bf16=True)
    u, _ = cx.static_solve(pdx.solve_opts(precond=pdx.PDX_PREC_LEARNED, tol=1e-8))
    return dict(loss=loss, grad=grad, M=M, u=u)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _counts(case):
    """(d, nodes, elements, PD nodes, blocks of K) of the case's mesh, the crack's own PD nodes left out."""
    if case["mesh"] in ("box", "penny"):
        n, pd = case["n"], case["pd"]
        return 3, n ** 3, (n - 1) ** 3, pd ** 3, 27 * (n ** 3 - pd ** 3) + 123 * pd ** 3
    nx, ny = case["nx"], case["ny"]
    pd = int(nx * ny * 0.2) if case["mesh"] == "plate" else 20 * nx // 4
    return 2, nx * ny, (nx - 1) * (ny - 1), pd, 9 * (nx * ny - pd) + 29 * pd


def work(case):
    kind = case["kind"]
    if kind == "families":
        f, bonds = case["n"] ** 3, case["n"] ** 3 * 115
        return dict(bytes=f * (40 + 2 * 81 * 8) + bonds * (4 + 36), flops=bonds * (135 + 162) + f * (243 + 1458))
    d, nn, ne, npd, nblk = _counts(case)
    nen = 8 if d == 3 else 4
    dof, matvec = nn * d, 2.0 * d * d * nblk
    geometry = nn * 24 + ne * nen * 4
    # element blocks: M = sum_g w g g^T per node pair and Gauss point; bonds: shape tensor, one solve, the block
    p = 9 if d == 3 else 5
    assembly = ne * nen * nen * (nen + 1) / 2 * 2 * d * d + (nblk / nn) * npd * (4 * p * p + 2 * d * d)
    if kind == "explicit":
        # a step reads u_n, u_{n-1}, the mass and the load and writes u_{n+1}; the consistent mass is solved by some 20
        # products at least
        return dict(bytes=geometry + case["steps"] * dof * 40, flops=case["steps"] * matvec * (1 if case["lumped"] else 10))
    if kind == "static":
        return dict(bytes=geometry + dof * 16, flops=assembly + 60 * matvec)
    if kind == "newmark":
        return dict(bytes=geometry + case["steps"] * dof * 64, flops=assembly + case["steps"] * 60 * matvec)
    if kind == "loadstep":
        return dict(bytes=geometry + dof * 24 + nn * 48, flops=assembly + matvec + ne * nen * 400)
    if kind == "csr":
        return dict(bytes=geometry + nblk * d * d * 16 + dof * 16, flops=assembly + 600 * matvec)
    g = case["probes"] * 6 * matvec + 3 * nn * 4 * 2 * 2 * 32 * 32
    return dict(bytes=geometry + nblk * d * d * 8 + dof * 16, flops=g + 100 * matvec)


def tolerance(case):
    """About four times what plain FP64 torch (exact) differs by, over the sizes above, rounded up to a power of ten."""
    kind = case["kind"]
    if kind == "families":
        return dict(rel=1e-7, max=1e-5)  # FP32 bond blocks
    if kind == "explicit":
        return dict(rel=1e-7, max=1e-5) if case["fp32"] else dict(rel=1e-12, max=1e-10)
    if kind == "loadstep":
        return dict(rel=1e-11, max=1e-9)  # K u of a smooth field cancels, more on finer meshes
    if kind == "newmark":
        return dict(rel=1e-6, max=1e-4)  # solves to a 1e-8 residual
    if kind == "learned":
        return dict(rel=1e-2, max=0.5)  # BF16 activations in the smoother
    return dict(rel=1e-5, max=1e-3)  # a 1e-8 residual (csr 1e-10) times the conditioning of a static system


# ---------------------------------------------------------------------------
# the same results in plain torch, FP64
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _t(a, dtype=None):
    t = torch.as_tensor(np.ascontiguousarray(a))
    return t.to(_dev(), dtype if dtype is not None else (torch.float64 if t.is_floating_point() else torch.int64))


_GP = 1.0 / math.sqrt(3.0)
_S8 = np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1], [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]], float)
_S4 = np.array([[-1, -1], [1, -1], [1, 1], [-1, 1]], float)


def _shape(points, corners):
    """Shape functions [g, a] and parent derivatives [g, a, d] of the (bi/tri)linear element at the points [g, d]."""
    f = 1 + points[:, None, :] * corners[None]
    d = corners.shape[1]
    N = f.prod(2) / 2 ** d
    dN = np.stack([corners[None, :, i] * np.delete(f, i, 2).prod(2) / 2 ** d for i in range(d)], 2)
    return _t(N), _t(dN)


def _basis(xi):
    x = xi.unbind(-1)
    if len(x) == 2:
        return torch.stack([x[0], x[1], x[0] ** 2, x[1] ** 2, x[0] * x[1]], -1)
    return torch.stack([*x, x[0] ** 2, x[1] ** 2, x[2] ** 2, x[0] * x[1], x[1] * x[2], x[2] * x[0]], -1)


def _bond_blocks(lam, mu, s, w):
    """Bond stiffness [.., d, d] from the second-order part s of the per-bond solution and the bond weight w."""
    if s.shape[-1] == 3:
        g = [(2 * mu + lam) * s[..., 0] + mu * s[..., 1], (lam + mu) * s[..., 2], (lam + mu) * s[..., 2],
             (2 * mu + lam) * s[..., 1] + mu * s[..., 0]]
        d = 2
    else:
        tr = s[..., 0] + s[..., 1] + s[..., 2]
        dg = [(mu + lam) * s[..., i] + mu * tr for i in range(3)]
        xy, yz, zx = ((lam + mu) * s[..., 3 + i] for i in range(3))
        g, d = [dg[0], xy, zx, xy, dg[1], yz, zx, yz, dg[2]], 3
    return torch.stack(g, -1).reshape(*s.shape[:-1], d, d) * w[..., None, None]


def _solve_bonds(xi, w, fam, nfam):
    """Per bond the solution of its family's shape-tensor system (A x = p, A = S diag(s)) and the families' S."""
    p = _basis(xi)
    n, d = p.shape[1], xi.shape[1]
    S = torch.zeros(nfam, n, n, dtype=torch.float64, device=xi.device)
    for i in range(0, len(p), 1 << 21):
        q = p[i:i + (1 << 21)]
        S.index_add_(0, fam[i:i + (1 << 21)], q[:, :, None] * (q * w[i:i + (1 << 21), None])[:, None, :])
    half = torch.ones(n, dtype=torch.float64, device=xi.device)
    half[d:2 * d] = 0.5
    # rows and columns scaled to the family's size before the inverse, so that it is well conditioned
    sc = S.diagonal(dim1=1, dim2=2).sqrt()
    inv = torch.linalg.inv(S / sc[:, :, None] / sc[:, None, :]) / sc[:, :, None] / sc[:, None, :]
    x = torch.cat([torch.matmul(inv[fam[i:i + (1 << 21)]], p[i:i + (1 << 21), :, None])[..., 0]
                   for i in range(0, len(p), 1 << 21)])
    return x / half, S, half


def _segments_cross(a1, a2, b1, b2):
    lo, hi = np.minimum, np.maximum
    box = ((hi(a1[:, 0], a2[:, 0]) < min(b1[0], b2[0])) | (hi(a1[:, 1], a2[:, 1]) < min(b1[1], b2[1]))
           | (max(b1[0], b2[0]) < lo(a1[:, 0], a2[:, 0])) | (max(b1[1], b2[1]) < lo(a1[:, 1], a2[:, 1])))
    s1 = (((a1[:, 0] - b1[0]) * (b2[1] - b1[1]) - (a1[:, 1] - b1[1]) * (b2[0] - b1[0]))
          * ((a2[:, 0] - b1[0]) * (b2[1] - b1[1]) - (a2[:, 1] - b1[1]) * (b2[0] - b1[0])))
    s2 = (((b1[0] - a1[:, 0]) * (a2[:, 1] - a1[:, 1]) - (b1[1] - a1[:, 1]) * (a2[:, 0] - a1[:, 0]))
          * ((b2[0] - a1[:, 0]) * (a2[:, 1] - a1[:, 1]) - (b2[1] - a1[:, 1]) * (a2[:, 0] - a1[:, 0])))
    return ~box & ~((s1 > 0) | (s2 > 0))


def _cross(u, v):
    return np.stack([u[..., 1] * v[..., 2] - u[..., 2] * v[..., 1], u[..., 2] * v[..., 0] - u[..., 0] * v[..., 2],
                     u[..., 0] * v[..., 1] - u[..., 1] * v[..., 0]], -1)


def _dot(u, v):
    return u[..., 0] * v[..., 0] + u[..., 1] * v[..., 1] + u[..., 2] * v[..., 2]


def _segments_cut_triangle(p1, p2, T):
    n = _cross(T[1] - T[0], T[2] - T[0])
    t = _dot(p1 - T[0], n) * _dot(p2 - T[0], n)
    with np.errstate(all="ignore"):
        X = p1 + (_dot(T[0] - p1, n) / _dot(p2 - p1, n))[:, None] * (p2 - p1)
        area = lambda u, v: np.sqrt(_dot(_cross(u, v), _cross(u, v)))  # noqa: E731
        A = math.sqrt(_dot(n, n))
        Ap = area(T[1] - X, T[2] - X) + area(X - T[0], T[2] - T[0]) + area(T[1] - T[0], X - T[0])
        return (t == 0) | ((t < 0) & ~(np.abs(Ap - A) > A * 1.0e-14))


class _Plain:
    """The discrete system of a mesh on a logical grid: element stiffnesses, bond blocks, masses, loads."""

    def __init__(self, case, mesh):
        self.mesh, self.d = mesh, mesh["dim"]
        d = self.d
        x = np.asarray(mesh["x"], float)
        self.nn, self.x = len(x), x
        E, nu = mesh["E"], mesh["nu"]
        self.mu = 0.5 * E / (1 + nu)
        self.lam = E * nu / (1 - nu * nu) if d == 2 else E * nu / ((1 - 2 * nu) * (1 + nu))
        nv = 3 if d == 2 else 6
        D = np.zeros((nv, nv))
        D[:d, :d] = self.lam
        D[np.arange(nv), np.arange(nv)] = [self.lam + 2 * self.mu] * d + [self.mu] * (nv - d)
        self.D = _t(D)
        self.free = np.ones(self.nn * d, bool)
        self.presc = np.zeros(self.nn * d)
        for s in mesh["ebc"]:
            at = (np.asarray(s["nid"]) - 1) * d + s["dof"]
            self.free[at] = False
            self.presc[at] = s["val"]
        self.freet = _t(self.free, torch.bool)
        # elements: volumes, node volumes, the crack's elements turned into PD elements
        self.nen = 8 if d == 3 else 4
        econ = np.asarray(mesh["econ"])[:, :self.nen].astype(np.int64) - 1
        self.corners = _S8 if d == 3 else _S4
        self.N, self.dN = _shape(self.corners * _GP, self.corners)
        J = torch.einsum("gai,eaj->egij", self.dN, _t(x[econ][:, :, :d]))
        ev = torch.linalg.det(J).sum(1).cpu().numpy()
        nvol = np.bincount(econ.ravel(), np.repeat(ev / self.nen, self.nen), self.nn)
        algo = np.asarray(mesh["algo"]).copy()
        cracks = np.asarray(mesh["cracks"], float).reshape(-1, 3, 3)
        for c in cracks:
            e = np.nonzero(algo == 2)[0]
            if d == 3:
                z = x[econ[e]][:, :, 2]
                e = e[(z.min(1) <= c[:, 2].max()) & (z.max(1) >= c[:, 2].min())]
            edges = [(i, (i + 1) % 4) for i in range(4)]
            if d == 3:
                edges += [(4 + i, 4 + (i + 1) % 4) for i in range(4)] + [(i, 4 + i) for i in range(4)]
            cut = np.zeros(len(e), bool)
            for i, j in edges:
                p, q = x[econ[e, i]], x[econ[e, j]]
                cut |= _segments_cross(p, q, c[0], c[1]) if d == 2 else _segments_cut_triangle(p, q, c)
            algo[e[cut]] = 1
        pd, fe = econ[algo == 1], econ[algo == 2]
        self.fe = _t(fe)
        self.mass_lumped = nvol * mesh["rho"]
        # families of the PD elements' nodes: nodes within either horizon
        fam = np.unique(pd)
        self.famid = np.full(self.nn, -1, np.int64)
        self.famid[fam] = np.arange(len(fam))
        fv = np.bincount(pd.ravel(), np.repeat(ev[algo == 1] / self.nen, self.nen), self.nn)[fam]
        hz = mesh["fac"] * nvol ** (1.0 / d)
        dims = (case["n"],) * 3 if d == 3 else (case["nx"], case["ny"])
        tiny = ev.min() ** (2.0 / d) * 1e-16
        ki, ji = [], []
        grid = [(fam // int(np.prod(dims[:i]))) % dims[i] for i in range(d)]
        for o in np.ndindex(*(9,) * d):
            at = [grid[i] + o[i] - 4 for i in range(d)]
            ok = np.all([(at[i] >= 0) & (at[i] < dims[i]) for i in range(d)], 0)
            k = np.nonzero(ok)[0]
            j = sum(at[i][k] * int(np.prod(dims[:i])) for i in range(d))
            r2 = ((x[j] - x[fam[k]]) ** 2).sum(1)
            near = (r2 > tiny) & ((r2 < hz[fam[k]] ** 2 + tiny) | (r2 < hz[j] ** 2 + tiny))
            ki.append(k[near])
            ji.append(j[near])
        ki, ji = np.concatenate(ki), np.concatenate(ji)
        intact = np.ones(len(ki), bool)
        for c in cracks:
            p, q = x[fam[ki]], x[ji]
            intact &= ~(_segments_cross(p, q, c[0], c[1]) if d == 2 else _segments_cut_triangle(p, q, c))
        xi = _t((x[ji] - x[fam[ki]])[:, :d])
        delta = _t(hz[fam])
        self.bond_fam, self.bond_node, self.fam_node = _t(ki), _t(ji), _t(fam)
        w = torch.exp(-(xi ** 2).sum(1) / mesh["nlf"] ** 2 / delta[self.bond_fam] ** 2) * _t(nvol[ji])
        s, _, _ = _solve_bonds(xi, w, self.bond_fam, len(fam)) if len(ki) else (xi.new_zeros(0, 5 if d == 2 else 9), 0, 0)
        w = w * _t(intact.astype(float))
        self.fam_v = _t(fv)
        self.H = -_bond_blocks(self.lam, self.mu, s[:, d:], w) * self.fam_v[self.bond_fam][:, None, None]
        self.c = s[:, :d] * w[:, None]  # strain weights of the bonds
        # boundary of the PD region: tractions N D C of the family of each boundary node
        if d == 2:
            f = np.concatenate([pd[:, [i, (i + 1) % 4]] for i in range(4)])
        else:
            f = [(0, 1, 2, 3), (4, 5, 6, 7), (0, 3, 7, 4), (1, 2, 6, 5), (0, 4, 5, 1), (3, 7, 6, 2)]
            f = np.concatenate([pd[:, list(q)] for q in f])
            sense = np.repeat([-1, 1, -1, 1, -1, 1], len(pd))
            first = f.argmin(1)
            f = f[np.arange(len(f))[:, None], (first[:, None] + np.arange(4)) % 4]
            f = np.where(sense[:, None] < 0, f[:, ::-1], f)
        _, inv, cnt = np.unique(np.sort(f, 1), axis=0, return_inverse=True, return_counts=True)
        f = f[cnt[inv.ravel()] == 1]
        if d == 2:
            nx, ny = x[f[:, 1], 1] - x[f[:, 0], 1], x[f[:, 0], 0] - x[f[:, 1], 0]
            z = 0 * nx
            Nm = 0.5 * np.stack([nx, z, ny, z, ny, nx], 1).reshape(-1, 2, 3)
        else:
            n1 = np.cross(x[f[:, 1]] - x[f[:, 0]], x[f[:, 2]] - x[f[:, 0]])
            n2 = np.cross(x[f[:, 3]] - x[f[:, 0]], x[f[:, 2]] - x[f[:, 0]])
            a1, a2 = np.linalg.norm(n1, axis=1), np.linalg.norm(n2, axis=1)
            n = n1 / a1[:, None] * ((a1 + a2) * 0.5 * 0.25)[:, None]
            z = 0 * a1
            Nm = np.stack([n[:, 0], z, z, n[:, 1], z, n[:, 2], z, n[:, 1], z, n[:, 0], n[:, 2], z, z, z, n[:, 2], z,
                           n[:, 1], n[:, 0]], 1).reshape(-1, 3, 6)
        ND = np.zeros((len(fam), d, nv))
        for a in range(f.shape[1]):
            np.add.at(ND, self.famid[f[:, a]], Nm)
        self.H = self.H + torch.matmul((_t(ND) @ self.D)[self.bond_fam], self._strain_blocks(self.c))
        # element stiffness: B^T D B w detJ over the Gauss points
        self.Ke = torch.zeros(len(fe), self.nen * d, self.nen * d, dtype=torch.float64, device=_dev())
        for i in range(0, len(fe), 1 << 17):
            J = torch.einsum("gai,eaj->egij", self.dN, _t(x[fe[i:i + (1 << 17)]][:, :, :d]))
            B = self._strain_blocks(torch.einsum("egij,gaj->egai", torch.linalg.inv(J), self.dN))  # [e, g, a, nv, d]
            B = B.transpose(2, 3).reshape(B.shape[0], B.shape[1], nv, self.nen * d)
            w = torch.linalg.det(J)[..., None, None]
            self.Ke[i:i + (1 << 17)] = (B.transpose(2, 3) @ (self.D @ B) * w).sum(1)
        # loads of the natural boundary conditions for a unit traction
        self.f_unit = []
        for s in mesh["nbc"]:
            con = np.asarray(s["con"]).astype(np.int64) - 1
            if d == 2:
                t = x[con[:, 1]] - x[con[:, 0]]
                fe_ = np.repeat((0.5 * np.stack([t[:, 1], -t[:, 0]], 1))[:, None], 2, 1)
            else:
                N, dN = (v.cpu().numpy() for v in _shape(_S4 * _GP, _S4))
                g = np.einsum("gai,eaj->egij", dN, x[con])
                fe_ = np.einsum("ga,egj->eaj", N, np.cross(g[:, :, 0], g[:, :, 1]))
            f_ = np.zeros((self.nn, d))
            np.add.at(f_, con, fe_)
            self.f_unit.append(_t(f_.ravel()))

    def _strain_blocks(self, c):
        """Strain operator blocks [.., nv, d] of the weights c [.., d]: (xx, yy, xy) or (xx, yy, zz, xy, yz, zx)."""
        z = torch.zeros_like(c[..., 0])
        if self.d == 2:
            a, b = c.unbind(-1)
            m = [a, z, z, b, b, a]
        else:
            a, b, e = c.unbind(-1)
            m = [a, z, z, z, b, z, z, z, e, b, a, z, z, e, b, e, z, a]
        return torch.stack(m, -1).reshape(*c.shape[:-1], len(m) // self.d, self.d)

    def load(self, scale):
        f = torch.zeros(self.nn * self.d, dtype=torch.float64, device=_dev())
        for s, u in zip(scale, self.f_unit):
            f += s * u
        return f

    def mul(self, u):
        """K u over all DOFs."""
        U = u.reshape(self.nn, self.d)
        y = torch.zeros_like(U)
        if len(self.fe):
            r = torch.matmul(self.Ke, U[self.fe].reshape(len(self.fe), -1, 1))
            y.index_add_(0, self.fe.reshape(-1), r.reshape(-1, self.d))
        k = self.fam_node[self.bond_fam]
        y.index_add_(0, k, torch.matmul(self.H, (U[self.bond_node] - U[k])[:, :, None])[..., 0])
        return y.reshape(-1)

    def diag_blocks(self):
        B = torch.zeros(self.nn, self.d, self.d, dtype=torch.float64, device=_dev())
        for a in range(self.nen if len(self.fe) else 0):
            i = slice(a * self.d, (a + 1) * self.d)
            B.index_add_(0, self.fe[:, a], self.Ke[:, i, i])
        B.index_add_(0, self.fam_node[self.bond_fam], -self.H)
        return B

    def mass(self):
        """Consistent mass: element matrices [fe, a, b] and the lumped PD part per node."""
        m = torch.zeros(len(self.fe), self.nen, self.nen, dtype=torch.float64, device=_dev())
        NN = self.N[:, :, None] * self.N[:, None, :]
        for i in range(0, len(self.fe), 1 << 17):
            J = torch.einsum("gai,eaj->egij", self.dN, _t(self.x)[self.fe[i:i + (1 << 17)]][:, :, :self.d])
            m[i:i + (1 << 17)] = torch.einsum("eg,gab->eab", torch.linalg.det(J) * self.mesh["rho"], NN)
        pd = torch.zeros(self.nn, dtype=torch.float64, device=_dev())
        pd[self.fam_node] = self.fam_v * self.mesh["rho"]
        return m, pd

    def mass_mul(self, m, pd, u):
        U = u.reshape(self.nn, self.d)
        y = U * pd[:, None]
        y.index_add_(0, self.fe.reshape(-1), torch.matmul(m, U[self.fe]).reshape(-1, self.d))
        return y.reshape(-1)

    def mass_diag(self, m, pd):
        v = pd.clone()
        return v.index_add_(0, self.fe.reshape(-1), m.diagonal(dim1=1, dim2=2).reshape(-1))

    def solve(self, mul, blocks, b, tol=1e-14, most=60000):
        """Masked system solved by BiCGStab with node blocks, restarted on the true residual down to rounding."""
        free = self.freet.reshape(self.nn, self.d)
        eye = torch.eye(self.d, dtype=torch.float64, device=_dev())
        inv = torch.linalg.inv(torch.where(free[:, :, None] & free[:, None, :], blocks, eye))
        A = lambda v: torch.where(self.freet, mul(v), 0.0)  # noqa: E731
        P = lambda v: torch.where(self.freet, torch.matmul(inv, v.reshape(self.nn, self.d, 1)).reshape(-1), 0.0)  # noqa: E731
        b = torch.where(self.freet, b, 0.0)
        bn = float(b.norm())
        x, done, last = torch.zeros_like(b), 0, math.inf
        while bn > 0 and done < most:
            r = b - A(x)
            now = float(r.norm()) / bn
            if now < tol or now > 0.5 * last:
                break
            last = now
            rh, rho, al, om = r.clone(), 1.0, 1.0, 1.0
            p, v, y, goal = torch.zeros_like(r), torch.zeros_like(r), torch.zeros_like(r), now * 1e-7 * bn
            best, at = math.inf, y
            for it in range(most - done):
                rho1 = rh @ r
                p = r + (rho1 / rho * (al / om)) * (p - om * v) if it else r.clone()
                ph = P(p)
                v = A(ph)
                rho, al = rho1, rho1 / (rh @ v)
                s = r - al * v
                sh = P(s)
                t = A(sh)
                om = (t @ s) / (t @ t)
                y = y + al * ph + om * sh
                r = s - om * t
                if it % 25 == 24:
                    n = float(r.norm())
                    if n < best:
                        best, at = n, y
                    if n < goal or not math.isfinite(n) or n > 1e4 * best:
                        break
            done += it + 1
            x = x + at
        return x

    def stresses(self, u):
        d, nv = self.d, 3 if self.d == 2 else 6
        U = u.reshape(self.nn, d)
        k = self.fam_node[self.bond_fam]
        e = torch.matmul(self._strain_blocks(self.c), (U[self.bond_node] - U[k])[:, :, None])[..., 0]
        eps = torch.zeros(len(self.fam_node), nv, dtype=torch.float64, device=_dev()).index_add_(0, self.bond_fam, e)
        out = torch.zeros(self.nn, nv, dtype=torch.float64, device=_dev())
        out[self.fam_node] = eps @ self.D
        n = torch.zeros(self.nn, dtype=torch.float64, device=_dev())
        n[self.fam_node] = 1
        # Gauss-point stresses extrapolated to the corners; the quadrilateral's points are taken in the order
        # (-,-), (+,-), (-,+), (+,+) while its extrapolation counts them around the element
        L = _shape(self.corners * math.sqrt(3.0), self.corners)[0]
        order = [0, 1, 3, 2] if d == 2 else list(range(8))
        for i in range(0, len(self.fe), 1 << 17):
            con = self.fe[i:i + (1 << 17)]
            J = torch.einsum("gai,eaj->egij", self.dN, _t(self.x)[con][:, :, :d])
            g = torch.einsum("egij,gaj->egai", torch.linalg.inv(J), self.dN)
            sg = torch.matmul(self._strain_blocks(g), U[con][:, None, :, :, None])[..., 0].sum(2) @ self.D
            out.index_add_(0, con.reshape(-1), torch.einsum("ag,egv->eav", L, sg[:, order]).reshape(-1, nv))
            n.index_add_(0, con.reshape(-1), torch.ones(con.numel(), dtype=torch.float64, device=_dev()))
        out = out / n[:, None].clamp(min=1)
        full = torch.zeros(self.nn, 6, dtype=torch.float64, device=_dev())
        full[:, [0, 1, 3] if d == 2 else list(range(6))] = out
        return full

    def csr(self):
        """Values of K_ff, rows and columns in equation order (every stored block, broken bonds as zeros)."""
        d = self.d
        eq = torch.cumsum(self.freet, 0) - 1
        neq = int(self.freet.sum())
        fe = (self.fe[:, :, None] * d + torch.arange(d, device=_dev())).reshape(len(self.fe), -1)
        k, j = self.fam_node[self.bond_fam], self.bond_node
        self_ = torch.zeros(len(self.fam_node), d, d, dtype=torch.float64, device=_dev()).index_add_(0, self.bond_fam, -self.H)
        blocks = torch.cat([self.H, self_])
        bk, bj = torch.cat([k, self.fam_node]), torch.cat([j, self.fam_node])
        i = torch.arange(d, device=_dev())
        row = torch.cat([fe[:, :, None].expand_as(self.Ke).reshape(-1),
                         (bk[:, None, None] * d + i[None, :, None]).expand_as(blocks).reshape(-1)])
        col = torch.cat([fe[:, None, :].expand_as(self.Ke).reshape(-1),
                         (bj[:, None, None] * d + i[None, None, :]).expand_as(blocks).reshape(-1)])
        val = torch.cat([self.Ke.reshape(-1), blocks.reshape(-1)])
        ok = self.freet[row] & self.freet[col]
        key, inv = torch.unique(eq[row[ok]] * neq + eq[col[ok]], return_inverse=True)
        return torch.zeros(len(key), dtype=torch.float64, device=_dev()).index_add_(0, inv, val[ok])


def _exact_families(case, seed):
    c, lam, mu = _cloud(case, seed)
    x, n, delta = c["x"], case["n"], c["delta"]
    cs, lo = delta.max(), x.min(0)
    nb = np.maximum(1, np.floor((x.max(0) - lo) / cs).astype(np.int64) + 1)
    cell = np.clip(np.floor((x - lo) / cs).astype(np.int64), 0, nb - 1)
    tiny = delta.min() ** 2 * 1e-16
    grid = [(np.arange(n ** 3) // n ** i) % n for i in range(3)]
    ks, js = [], []
    for o in np.ndindex(9, 9, 9):
        at = [grid[i] + o[i] - 4 for i in range(3)]
        k = np.nonzero(np.all([(a >= 0) & (a < n) for a in at], 0))[0]
        j = sum(at[i][k] * n ** i for i in range(3))
        r2 = ((x[j] - x[k]) ** 2).sum(1)
        near = (r2 > tiny) & ((r2 < delta[k] ** 2 + tiny) | (r2 < delta[j] ** 2 + tiny))
        ks.append(k[near])
        js.append(j[near])
    ks, js = np.concatenate(ks), np.concatenate(js)
    # members in cell order (x outermost), each cell's nodes in node order
    o = np.lexsort((js, cell[js, 2], cell[js, 1], cell[js, 0], ks))
    k, j = _t(ks[o]), _t(js[o])
    X, dl = _t(x), _t(delta)
    xi = X[j] - X[k]
    w = torch.exp(-(xi ** 2).sum(1) / _NLF ** 2 / dl[k] ** 2) * _t(c["vol"])[j]
    s, S, half = _solve_bonds(xi, w, k, n ** 3)
    G = _bond_blocks(lam, mu, s[:, 3:], w).reshape(-1, 9)
    # the self block leads each family's members
    start = torch.searchsorted(k, torch.arange(n ** 3, device=k.device)) + torch.arange(n ** 3, device=k.device)
    H = torch.zeros(len(k) + n ** 3, 9, dtype=torch.float64, device=k.device)
    H[torch.arange(len(k), device=k.device) + k + 1] = G
    H[start] = -torch.zeros(n ** 3, 9, dtype=torch.float64, device=k.device).index_add_(0, k, G)
    sc = S.diagonal(dim1=1, dim2=2).sqrt()
    L = torch.linalg.cholesky(S / sc[:, :, None] / sc[:, None, :]) * sc[:, :, None]
    return dict(A=(S * half).cpu().numpy(), L=L.cpu().numpy(), H=H.cpu().numpy())


def exact(case, seed):
    kind = case["kind"]
    if kind == "families":
        return _exact_families(case, seed)
    mesh = _mesh(case, seed)
    S = _Plain(case, mesh)
    out = lambda v: v[S.freet].cpu().numpy()  # noqa: E731
    zero = torch.zeros(S.nn * S.d, dtype=torch.float64, device=_dev())
    up = _t(S.presc)
    load = [s["val"] for s in mesh["nbc"]]
    dt = mesh["dt"]
    if kind == "explicit":
        f = S.load(load)
        if case["lumped"]:
            m = _t(np.repeat(S.mass_lumped, S.d))
            acc = lambda F: F / m  # noqa: E731
        else:
            me, pd = S.mass()
            blocks = torch.diag_embed(S.mass_diag(me, pd)[:, None].expand(-1, S.d))
            acc = lambda F: S.solve(lambda v: S.mass_mul(me, pd, v), blocks, F, 1e-15)  # noqa: E731
        a = up.clone()
        b = a + torch.where(S.freet, acc(f - S.mul(a)) * (0.5 * dt * dt), 0.0)
        for _ in range(case["steps"]):
            a, b = b, torch.where(S.freet, 2 * b - a + dt * dt * acc(f - S.mul(b)), b)
        return dict(u=out(b), u_prev=out(a))
    if kind == "loadstep":
        u = _t(_field(mesh, seed))
        return dict(F=out(S.load(load) - S.mul(u)), sigma=S.stresses(u).cpu().numpy())
    if kind == "newmark":
        beta, gamma = mesh["beta"], mesh["gamma"]
        me, pd = S.mass()
        blocks = S.diag_blocks() * (beta * dt * dt) + torch.diag_embed(S.mass_diag(me, pd)[:, None].expand(-1, S.d))
        eff = lambda v: S.mass_mul(me, pd, v) + beta * dt * dt * S.mul(v)  # noqa: E731
        u, v, a, rate, val = zero, zero, zero, torch.zeros_like(zero), up.clone()
        for s in mesh["ebc"]:
            if s.get("vary"):
                rate[_t((np.asarray(s["nid"]) - 1) * S.d + s["dof"])] = dt * s["vel"]
        for i in range(case["steps"]):
            un = torch.where(S.freet, u + dt * v + dt * dt * (0.5 - beta) * a, val + rate)
            f = S.load([s["val"] + (i * dt * s["vel"] if s.get("vary") else 0.0) for s in mesh["nbc"]])
            a1 = S.solve(eff, blocks, f - S.mul(un))
            u = u + dt * v + dt * dt * ((0.5 - beta) * a + beta * a1)
            v = v + dt * ((1 - gamma) * a + gamma * a1)
            a, val = a1, val + rate
        return dict(u=out(u), v=out(v), a=out(a))
    F = S.load(load) - S.mul(up)
    if kind == "static":
        return dict(F=out(F), u=out(S.solve(S.mul, S.diag_blocks(), F, 1e-12)))
    if kind == "csr":
        return dict(K=S.csr().cpu().numpy(), F=out(F), x=out(S.solve(S.mul, S.diag_blocks(), F, 1e-12)))
    # the probes are the library's own random vectors, and the smoother is a BF16 network's
    return dict(loss=None, grad=None, M=None, u=out(S.solve(S.mul, S.diag_blocks(), F, 1e-12)))
