"""Bounded directions whose ghost cells the caller keeps (boundary code 0,
interior): a forward Euler step of one array over the domain reads the caller's
value in every such ghost cell, those beside a periodic boundary included, and
not the value a periodic image of it holds.  The fused stages against the
pass-structured kernels, bit for bit, with other random values in every ghost
cell."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


BCS = {
    "y kept": ((1, 0, 1), (0, 0, 0), (0, 0, 0)),
    "y kept below, outflow above": ((1, 0, 1), (0, 0, 0), (0, 2, 0)),
    "x kept, z slip": ((0, 1, 0), (0, 0, 4), (0, 0, 4)),
    "y outflow": ((1, 0, 1), (0, 2, 0), (0, 2, 0)),
}


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("bc", list(BCS))
def test_kept_ghost_cells(ctx, bc, order):
    from amrsolver_amd import level as L
    print(f"case int_dir {bc} keep{order}", flush=True)
    n = (32, 28, 12)
    cls = P.closures_reference()
    per, lo, hi = BCS[bc]
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), per, lo_bc=lo, hi_bc=hi)
    lev = L.Level(g, P.decompose(n, (16, 28, 12)), cls, P.scheme(flux_euler=1, order_keep=order, visc=True, order_rk=1, stages_rk=1),
                  ctx=ctx)
    u = P.smooth_random_state(cls, n, 6)
    out = []
    for tiling, form in (((-1, 0, 0), 0), ((16, 16, 8), 1)):
        S = lev.new_state(layout="level")
        full = P.smooth_random_state(cls, tuple(reversed(S.tensors[0].shape[1:])), 7)
        S.upload_ghosted(full)
        S.upload(u)
        lev.set_tiling(*tiling, form=form)
        lev.advance(S, 0.0, 1e-6)
        out.append(S.download())
    lev.set_tiling(0)
    assert np.isfinite(out[1]).all()
    assert np.array_equal(out[0], out[1])
