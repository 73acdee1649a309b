"""Products of the consistent mass through its scalar node-pair values where the launch changes shape:
fewer nodes than workgroups, exactly as many, one more, quads, triangles with tetrahedra, and rows of
PD nodes longer than one pass of a row's lanes.  The explicit trajectory (one CG solve with M a step, to
1e-13) against the oracle's factorised M; the bound is that of the ordinary sizes' trajectories."""
import numpy as np
import pytest

from helpers import load_oracle, load_pdx, one_quad, rel, tet_box_mesh, workloads

pytestmark = pytest.mark.gpu

O = load_oracle()
W = workloads()
pdx = load_pdx()


def _plate(nx, ny):
    m = W.plate2d(nx=nx, ny=ny, dx=1e-3, pd_x=(0.005, 0.011))
    m["ebc"][2].update(val=0.0, vel=0.05, vary=True)
    return dict(m, dt=5e-8)


def _box():
    m = W.box3d(n=9, pd_block=5)
    m["nbc"][0].update(vel=1e9, vary=True)
    return dict(m, dt=5e-8)


def _tets():
    m = tet_box_mesh()
    top = np.nonzero(m["x"][:, 2] > m["x"][:, 2].max() - 1e-9)[0] + 1
    m["ebc"].append(dict(nid=top.astype(np.int32), dof=2, val=0.0, vel=0.05, vary=True))
    return dict(m, dt=2e-8)


CASES = {"quad": one_quad, "plate_512": lambda: _plate(16, 32), "plate_513": lambda: _plate(19, 27),
         "tets": _tets, "box_pd": _box}


@pytest.mark.parametrize("name", sorted(CASES))
def test_mass_product_trajectory(name):
    mesh = dict(CASES[name](), lumped_mass=False)
    u0, up0, _ = O.Model(mesh).dynamic_run(12)
    u1, up1 = pdx.Context(pdx.Model(mesh)).explicit_run(12)
    assert np.abs(u0).max() > 0
    assert rel(u1, u0) <= 1e-10 and rel(up1, up0) <= 1e-10, (rel(u1, u0), rel(up1, up0))


def test_consistent_steps_build_no_tiles_and_time_no_forms():
    """A size at which lumped steps go through the element tiles: the consistent-mass step walks K in its one form, so
    it builds none.  The tuning is timed when it is asked for, for the precision that was stepped only."""
    mesh = W.box3d(n=30, pd_block=8)
    mesh["lumped_mass"] = False
    mesh["dt"] = 2e-8
    cx = pdx.Context(pdx.Model(mesh))
    assert cx.explicit_tuning_full(pdx.PDX_FP64)[8] == -1
    u = cx.explicit_run(3)[0]
    assert not any(cx.tile_counts().values())
    assert cx.explicit_tuning_full(pdx.PDX_FP32)[8] == -1 and not cx.explicit_tuning_full(pdx.PDX_FP32)[6].any()
    full = cx.explicit_tuning_full(pdx.PDX_FP64)
    assert 0 <= full[8] < pdx.EXPLICIT_FORMS and (full[6] > 0).all()
    assert np.array_equal(cx.explicit_run(0)[0], u)
