"""The products with hex8 elements and PD families without their blocks of K (csrc/hex.hip) against the walk of K
(explicit steps) and against the assembled K and mass on the host (solves).

Both sum the same terms in FP64 in another order, so a trajectory differs by rounding only: a product of a row of some
30 to 130 blocks of 3 x 3 carries at most about 400 roundings of 1.1e-16 of its absolute terms, 5e-14, and the
differences of 25 steps stay below 25 times that: 1e-12.  The meshes lie above the size from which the tiles are used.
"""
import numpy as np
import pytest

from helpers import load_pdx, rel, workloads

pytestmark = pytest.mark.gpu
pdx, W = load_pdx(), workloads()


def _dt(mesh):
    mesh["lumped_mass"] = True  # the consistent-mass step walks K
    mesh["dt"] = 2e-8  # 1 mm elements of steel-like stiffness: a fraction of the critical step
    mesh["nbc"][0].update(vel=1e12, vary=True)
    mesh["ebc"][0].update(vel=1e-3, vary=True)
    return mesh


def _shuffled(mesh, seed=0):
    """The same body with its nodes renumbered and every element started at another corner."""
    rng = np.random.default_rng(seed)
    p = rng.permutation(len(mesh["x"]))
    inv = np.argsort(p)
    e = inv[np.asarray(mesh["econ"]) - 1] + 1
    turn, tip = [1, 2, 3, 0, 5, 6, 7, 4], [3, 2, 6, 7, 0, 1, 5, 4]
    for k in range(len(e)):
        if mesh["algo"][k] == 2:  # the PD elements' faces are matched by their corner order
            for _ in range(rng.integers(4)):
                e[k] = e[k][turn]
            for _ in range(rng.integers(4)):
                e[k] = e[k][tip]
    mesh["x"], mesh["econ"] = np.asarray(mesh["x"])[p], e.astype(np.int32)
    for s in mesh["ebc"]:
        s["nid"] = inv[np.asarray(s["nid"]) - 1] + 1
    for s in mesh["nbc"]:
        s["con"] = inv[np.asarray(s["con"]) - 1] + 1
    return mesh


def _with_tets(mesh, share=0.02):
    """Some of the FE hexahedra split into five tetrahedra each."""
    rng = np.random.default_rng(1)
    econ, nen, algo = np.asarray(mesh["econ"]), np.asarray(mesh["nen"]), np.asarray(mesh["algo"])
    split = (algo == 2) & (rng.random(len(econ)) < share)
    five = [(0, 1, 2, 5), (0, 2, 3, 7), (0, 5, 7, 4), (2, 7, 5, 6), (0, 2, 7, 5)]
    t = np.zeros((5 * int(split.sum()), 8), np.int32)
    t[:, :4] = np.concatenate([econ[split][:, list(q)] for q in five])
    mesh["econ"] = np.concatenate([econ[~split], t])
    mesh["nen"] = np.concatenate([nen[~split], np.full(len(t), 4, np.int32)])
    mesh["algo"] = np.concatenate([algo[~split], np.full(len(t), 2, np.int32)])
    return mesh


def _plate(mesh, layers):
    """The lowest layers of elements of a box, loaded on the new top."""
    n, per = len(mesh["x"]), 79 * 79
    e = np.asarray(mesh["econ"])
    keep = (e <= (layers + 1) * per).all(1)
    mesh.update(x=np.asarray(mesh["x"])[:(layers + 1) * per], econ=e[keep], nen=mesh["nen"][keep], algo=mesh["algo"][keep])
    mesh["nbc"][0]["con"] = np.asarray(mesh["nbc"][0]["con"]) - n + (layers + 1) * per
    return mesh


CASES = {
    "pd_block": lambda: W.box3d(n=31, pd_block=9),
    "elements_only": lambda: W.box3d(n=29, pd_block=0),
    "shuffled": lambda: _shuffled(W.box3d(n=30, pd_block=8)),
    "with_tets": lambda: _with_tets(W.box3d(n=33, pd_block=8)),  # too many rows left to K: no tiles
    "few_tets": lambda: _with_tets(W.box3d(n=33, pd_block=8), 0.004),
    "plate": lambda: _plate(W.box3d(n=79, pd_block=0), 4),
    "penny_crack": lambda: W.penny3d(n=32, pd_block=8),
}


def _tiled(cx, model, name=""):
    """The products went through the tiles, which hold every row that they may."""
    n = cx.tile_counts()
    if name == "with_tets":
        assert not any(n.values())
        return
    assert n["products"] > 0 and n["tiles"] > 0 and n["elements"] >= (model.nfe if name != "few_tets" else 1)
    assert (n["families"] > 0) == (model.nfam > 0)
    if not model.npde:
        assert n["rows"] == 0


@pytest.mark.parametrize("name", list(CASES))
def test_explicit_through_tiles_equals_walk_of_K(name):
    model = pdx.Model(_dt(CASES[name]()))
    tiles, walk = pdx.Context(model), pdx.Context(model)
    walk.explicit_set_form(pdx.PDX_FP64, 0)
    for steps in (1, 24):
        (u, up), (v, vp) = tiles.explicit_run(steps), walk.explicit_run(steps)
        assert np.linalg.norm(v) > 0
        assert rel(u, v) <= 1e-12 and rel(up, vp) <= 1e-12
    # the sums have one order: eager steps of another context give the same bits as the replayed ones
    eager = pdx.Context(model)
    eager.explicit_steps(25, use_graph=False)
    assert np.array_equal(eager.explicit_run(0)[0], u)
    # a form can still be set, and taken back, between steps; the tuning is reported as before
    tiles.explicit_set_form(pdx.PDX_FP64, 21)
    assert rel(tiles.explicit_run(6)[0], walk.explicit_run(6)[0]) <= 1e-12
    tiles.explicit_set_form(pdx.PDX_FP64, -1)
    assert rel(tiles.explicit_run(6)[0], walk.explicit_run(6)[0]) <= 1e-12
    _tiled(tiles, model, name)
    assert walk.tile_counts()["products"] == 0
    assert 0 <= tiles.explicit_tuning_full(pdx.PDX_FP64)[8] < pdx.EXPLICIT_FORMS
    assert rel(tiles.explicit_run(6)[0], walk.explicit_run(6)[0]) <= 1e-12


def test_fp32_force_through_tiles():
    """FP32 force (large models only): the tiles calculate in FP64, so they are no further from FP64 than the walk."""
    model = pdx.Model(_dt(W.box3d(n=65, pd_block=12)))
    ref, tiles, walk = (pdx.Context(model) for _ in range(3))
    ref.explicit_set_form(pdx.PDX_FP64, 0)
    walk.explicit_set_form(pdx.PDX_FP32, 0)
    u = ref.explicit_run(25)[0]
    e_tiles = rel(tiles.explicit_run(25, pdx.PDX_FP32)[0], u)
    e_walk = rel(walk.explicit_run(25, pdx.PDX_FP32)[0], u)
    assert e_tiles <= 1.2 * e_walk <= 1e-6
    _tiled(tiles, model)
    assert ref.tile_counts()["products"] == walk.tile_counts()["products"] == 0


def _csr(model, values):
    import scipy.sparse as sp
    ia, ja = model.csr()
    return sp.csr_matrix((values, ja, ia), shape=(model.neq, model.neq))


SOLVES = {"fp64": {}, "fp64_mirrored": {"mirrored": True}, "fp64_two_level": {"precond": 4}, "fp32_two_level": {"precision": 1, "precond": 4}}


@pytest.mark.parametrize("opts", list(SOLVES))
@pytest.mark.parametrize("name", list(CASES))
def test_solves_through_tiles(name, opts):
    """A Newmark step and a static solve: the residual of their results with the assembled matrices on the host, which
    the solver's own products come within rounding of (1e-8 asked for; 1e-11 for the products' rounding)."""
    mesh = _dt(CASES[name]())
    mesh["nbc"][0]["val"] = 1e6
    model = pdx.Model(mesh)
    cx = pdx.Context(model)
    K = _csr(model, cx.assemble(pdx.PDX_MODE_STATIC)[0])
    o = dict(precond=pdx.PDX_PREC_BLOCK_JACOBI, tol=1e-8)
    o.update(SOLVES[opts])
    _, _, a, st = cx.newmark_run(1, pdx.solve_opts(**o))
    keff = _csr(model, cx.mass_on_K()) + mesh["beta"] * mesh["dt"] ** 2 * K
    dU = model.values()  # u = v = a = 0: the predictor is the prescribed values, advanced
    for s in mesh["ebc"]:
        dU[(np.asarray(s["nid"]) - 1) * 3 + s["dof"]] += mesh["dt"] * s.get("vel", 0.0) * bool(s.get("vary", False))
    fresh = pdx.Context(model)
    F = fresh.assemble(pdx.PDX_MODE_NEWMARK, UN=dU)[1]
    assert np.linalg.norm(F - keff @ a) <= (1e-8 + 1e-11) * np.linalg.norm(F)
    assert st["converged"]
    u, st = fresh.static_solve(pdx.solve_opts(**o))
    if o.get("precision") == pdx.PDX_FP32:  # at these sizes FP32 products walk the blocks
        assert cx.tile_counts()["products"] == fresh.tile_counts()["products"] == 0
    else:
        _tiled(cx, model, name)
        _tiled(fresh, model, name)
    b = fresh.assemble(pdx.PDX_MODE_STATIC)[1]
    assert np.linalg.norm(b - K @ u) <= (1e-8 + 1e-11) * np.linalg.norm(b)


def test_fp32_two_level_through_tiles():
    """A static solve with FP32 vectors and the two-level preconditioner at a size where FP32 products go through the
    tiles; the residual is formed by another context's walk of K."""
    mesh = W.box3d(n=65, pd_block=12)
    model = pdx.Model(mesh)
    cx = pdx.Context(model)
    u, st = cx.static_solve(pdx.solve_opts(precision=pdx.PDX_FP32, precond=pdx.PDX_PREC_TWO_LEVEL, tol=1e-8))
    assert st["converged"] and st["refinements"] > 0
    _tiled(cx, model)
    walk = pdx.Context(model)
    b = walk.assemble(pdx.PDX_MODE_STATIC, want_K=False)[1]
    full, eq = model.values(), model.nodes()["eq"].ravel()
    full[eq >= 0] = u[eq[eq >= 0]]
    walk.set_dof_values(full)
    r = walk.assemble(pdx.PDX_MODE_EXPLICIT)[1]  # F_ext - K u
    assert walk.tile_counts()["products"] == 0
    assert np.linalg.norm(r) <= (1e-8 + 1e-11) * np.linalg.norm(b)


def test_several_natural_bc_sets_through_tiles():
    """Three traction sets (constant, ramped, on two faces) and a ramped prescribed face."""
    mesh = _dt(W.box3d(n=30, pd_block=8))
    n = 30
    nid = lambda i, j, k: i + n * (j + n * k) + 1
    side = [[nid(n - 1, j, k), nid(n - 1, j + 1, k), nid(n - 1, j + 1, k + 1), nid(n - 1, j, k + 1)]
            for j in range(n - 1) for k in range(n - 1)]
    top = np.asarray(mesh["nbc"][0]["con"])
    mesh["nbc"] = [dict(con=top[::2], val=3e5, vel=0.0, vary=False), dict(con=top, val=0.0, vel=2e12, vary=True),
                   dict(con=np.asarray(side, np.int32), val=-1e5, vel=1e12, vary=True)]
    model = pdx.Model(mesh)
    tiles, walk = pdx.Context(model), pdx.Context(model)
    walk.explicit_set_form(pdx.PDX_FP64, 0)
    for steps in (1, 13):
        assert rel(tiles.explicit_run(steps)[0], walk.explicit_run(steps)[0]) <= 1e-12
    tiles.assemble(pdx.PDX_MODE_STATIC, want_K=False)  # another K: the families' moments are formed again
    assert rel(tiles.explicit_run(7)[0], walk.explicit_run(7)[0]) <= 1e-12
    _tiled(tiles, model)


def test_fp32_newmark_through_tiles():
    """FP32 vectors with FP64 element arithmetic (large models only), refined: the same displacements as in FP64."""
    model = pdx.Model(_dt(W.box3d(n=65, pd_block=12)))
    run = []
    for p in (pdx.PDX_FP64, pdx.PDX_FP32):
        cx = pdx.Context(model)
        run.append(cx.newmark_run(2, pdx.solve_opts(precond=pdx.PDX_PREC_BLOCK_JACOBI, precision=p, tol=1e-10)))
    assert run[1][3]["converged"] and run[1][3]["refinements"] > 0
    _tiled(cx, model)
    for x, y in zip(run[0][:3], run[1][:3]):
        assert rel(y, x) <= 1e-8


@pytest.mark.parametrize("n, precision", [(65, pdx.PDX_FP32), (29, pdx.PDX_FP64)])
def test_newmark_with_beta_zero(n, precision):
    """beta = 0: the operator of a step is M alone (no K in it), above the sizes where its products go through the tiles.
    The acceleration solves M a = F to the tolerance asked for, checked with the assembled M."""
    mesh = _dt(W.box3d(n=n, pd_block=8))
    mesh["beta"] = 0.0
    mesh["nbc"][0]["val"] = 1e6
    model = pdx.Model(mesh)
    cx = pdx.Context(model)
    _, _, a, st = cx.newmark_run(1, pdx.solve_opts(precond=pdx.PDX_PREC_BLOCK_JACOBI, precision=precision, tol=1e-8))
    assert st["converged"]
    M = _csr(model, cx.mass_on_K())
    dU = model.values()
    for s in mesh["ebc"]:
        dU[(np.asarray(s["nid"]) - 1) * 3 + s["dof"]] += mesh["dt"] * s.get("vel", 0.0) * bool(s.get("vary", False))
    _tiled(cx, model)
    F = pdx.Context(model).assemble(pdx.PDX_MODE_NEWMARK, UN=dU)[1]
    assert np.linalg.norm(F - M @ a) <= (1e-8 + 1e-11) * np.linalg.norm(F)
