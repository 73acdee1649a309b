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
