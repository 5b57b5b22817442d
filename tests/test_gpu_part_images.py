"""A domain periodic in some directions and bounded in others, in one array:
the fused stages read the periodic images and fill only the ghost cells at the
physical boundaries.  Steps are bit for bit those of the pass-structured
kernels, which fill every ghost cell, with NaN in all ghost cells before the
first step; eager and captured."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


# periodic directions and boundary codes (2 foextrap, 3 symmetry, 4 slip, 5 no slip)
BCS = {
    "x bounded": ((0, 1, 1), (2, 0, 0), (2, 0, 0)),
    "y slip, no slip": ((1, 0, 1), (0, 4, 0), (0, 5, 0)),
    "z bounded": ((1, 1, 0), (0, 0, 3), (0, 0, 2)),
    "x and z bounded": ((0, 1, 0), (2, 0, 4), (3, 0, 2)),
}


def _run(lev, u, tiling, form):
    """Two eager and two captured steps on the level layout, NaN in the ghost
    cells at the start."""
    lev.set_tiling(*tiling, form=form) if form else lev.set_tiling(*tiling)
    S = lev.new_state(layout="level")
    S.tensors[0].fill_(float("nan"))
    S.upload(u)
    for _ in range(2):
        lev.advance(S, 0.0, 2e-7)
    a = S.download()
    for _ in range(2):
        lev.advance_graph(S, 2e-7, 1)
    b = S.download()
    lev.set_tiling(0)
    return a, b


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("n,mg", [((33, 20, 9), (33, 20, 9)), ((48, 34, 20), (32, 17, 12)), ((16, 16, 3), (16, 16, 3))])
@pytest.mark.parametrize("bc", list(BCS))
def test_part_images(ctx, bc, n, mg, order):
    from amrsolver_amd import level as L
    print(f"case part images {bc} {n} {mg} order {order}", flush=True)
    cls = P.closures_reference()
    per, lo, hi = BCS[bc]
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), per, lo_bc=lo, hi_bc=hi)
    lev = L.Level(g, P.decompose(n, mg), cls, P.scheme(flux_euler=1, order_keep=order, visc=True), ctx=ctx)
    u = P.smooth_random_state(cls, n, 6)
    ref = _run(lev, u, (-1, 0, 0), 0)
    for tz in (16, 2):
        got = _run(lev, u, (16, 16, tz), 1)
        assert np.isfinite(got[1]).all()
        assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1]), f"tz {tz}"


def test_part_images_walls(ctx):
    from amrsolver_amd import level as L
    n = (40, 33, 12)
    cls, g, _, parm = P.wall_channel(n)
    sch = P.scheme(flux_euler=1, order_keep=4, visc=True, source=True)
    lev = L.Level(g, P.decompose(n, (24, 17, 12)), cls, sch, ctx=ctx)
    lev.set_problem(wall_T=parm["Tw"], body_force_x=parm["fx"])
    u = P.wall_channel_state(cls, g, n, parm)
    out = []
    for tiling, form in (((-1, 0, 0), 0), ((16, 16, 5), 1)):
        print(f"case part images walls {tiling}", flush=True)
        lev.set_tiling(*tiling, form=form) if form else lev.set_tiling(*tiling)
        S = lev.new_state(layout="level")
        S.tensors[0].fill_(float("nan"))
        S.upload(u)
        for _ in range(3):
            lev.advance(S, 0.0, 2e-9)
        out.append(S.download())
        lev.set_tiling(0)
    assert np.isfinite(out[1]).all() and np.array_equal(out[0], out[1])
