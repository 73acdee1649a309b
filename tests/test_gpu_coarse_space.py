"""Coarse space of the two-level preconditioner (A P, the Galerkin matrix and its dense inverse) where the
launches change shape: one aggregate, one pivot block, an odd and an even count of 64-pivot blocks, rows
of A P that touch more aggregates than one pass of the kernel holds.

The probes of the learned smoother give y = K (I - Q K) z with Q = P (P^T K P)^-1 P^T on the free DOFs, so
P^T y = 0; P holds each aggregate's translations, hence every component of y sums to zero over the nodes.
y is stored in FP32: the sum is off by at most 2^-24 sum |y|, the inverse's FP64 error is small beside it."""
import numpy as np
import pytest

from helpers import load_pdx, workloads

pytestmark = pytest.mark.gpu

W = workloads()
pdx = load_pdx()


@pytest.mark.parametrize("dim, agg", [(2, 61), (2, 16), (2, 10), (2, 8), (2, 7), (2, 5), (2, 3), (2, 2),
                                      (3, 12), (3, 6), (3, 5), (3, 4), (3, 3), (3, 2)])
def test_coarse_correction_is_exact_on_translations(dim, agg):
    mesh = W.crack2d(seed=3, nx=61, ny=31, dx=0.1 / 60) if dim == 2 else W.box3d(n=12, pd_block=6)
    cx = pdx.Context(pdx.Model(mesh))
    cx.assemble(pdx.PDX_MODE_STATIC)
    y = pdx.gnn_inputs(cx, n_probes=3, probe_seed=agg, coarse_agg=agg)["y"].astype(np.float64).reshape(3, -1, dim)
    assert np.abs(y).max() > 0
    total, scale = np.abs(y.sum(1)), np.abs(y).sum(1)
    print(f"dim {dim} agg {agg}: {(total / scale).max():.1e}", flush=True)
    assert (total <= 2.0 ** -23 * scale).all(), (total / scale).max()


@pytest.mark.parametrize("n", [8, 9])
def test_aggregates_that_reach_512_others(n):
    """A PD body inside every node's horizon with one node per aggregate: each row of the Galerkin matrix holds all
    512 (one full list of the kernel) or 729 (two lists) aggregates.  The coarse space is then the whole space, so
    Q is K's inverse and y = K (I - Q K) z is rounding: with a condition number below 1e7 (1.0e6 for 729 nodes,
    asserted on the host), under 1e7 * 1e-16 * some 1e3 operations = 1e-6 of K's entries.  A lost 3 x 3 block
    column leaves 0.1."""
    import scipy.sparse as sp
    model = pdx.Model(W.box3d(n=n, pd_block=n, jitter=0.0, m=30.0))
    assert model.max_family == n ** 3
    cx = pdx.Context(model)
    ia, ja = model.csr()
    K = sp.csr_matrix((cx.assemble(pdx.PDX_MODE_STATIC)[0], ja, ia), shape=(model.neq, model.neq)).toarray()
    assert np.linalg.cond(K) < 1e7
    y = pdx.gnn_inputs(cx, n_probes=2, probe_seed=n, coarse_agg=1)["y"].astype(np.float64)
    ratio = np.abs(y).max() / np.abs(K).max()
    print(f"n {n}: {ratio:.1e}", flush=True)
    assert ratio <= 1e-6
