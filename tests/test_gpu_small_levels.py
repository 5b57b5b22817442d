"""Small levels: the CFL minimum over more boxes than box slots and over few
boxes, and stages on tiles of one and two planes.  Both are exact: a minimum
does not depend on its order, and a tile's plane count does not enter a
cell's arithmetic."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


@pytest.mark.parametrize("n,mg,cell", [((48, 48, 48), (4, 4, 4), (47, 46, 45)), ((48, 48, 48), (4, 4, 4), (1, 2, 3)),
                                       ((32, 24, 20), (16, 16, 16), (31, 3, 17)), ((40, 36, 20), (20, 36, 20), (5, 35, 0))])
def test_cfl_minimum_over_boxes(ctx, n, mg, cell):
    from amrsolver_amd import level as L
    print(f"case cfl {n} {mg} {cell}", flush=True)
    cls = P.closures_reference()
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    u = P.smooth_random_state(cls, n, 3)
    u[4][cell[2], cell[1], cell[0]] *= 4.0  # the hottest cell decides
    got = []
    for boxes in (P.decompose(n, mg), P.decompose(n, n)):
        lev = L.Level(g, boxes, cls, P.scheme(flux_euler=1, order_keep=4, visc=True), ctx=ctx)
        S = lev.new_state()
        S.upload(u)
        got.append(lev.est_time_step(S, 0.3))
    u[4][cell[2], cell[1], cell[0]] *= 0.25
    S.upload(u)
    assert got[0] == got[1] < lev.est_time_step(S, 0.3)


@pytest.mark.parametrize("order,visc", [(2, True), (4, True), (6, True), (4, False)])
@pytest.mark.parametrize("tz", [1, 2])
@pytest.mark.parametrize("layout", ["level", "boxes"])
def test_short_tiles(ctx, layout, tz, order, visc):
    from amrsolver_amd import level as L
    n = (33, 20, 7)
    print(f"case short tiles {n} tz {tz} order {order} visc {visc} {layout}", flush=True)
    cls = P.closures_reference()
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    lev = L.Level(g, P.decompose(n, (17, 20, 7)), cls, P.scheme(flux_euler=1, order_keep=order, visc=visc), ctx=ctx)
    u = P.smooth_random_state(cls, n, 3)
    for form in (0, 1) if visc and order < 6 else (0,):
        got = []
        for t in (tz, 16):
            lev.set_tiling(16, 16, t, form)
            S = lev.new_state(layout=layout)
            S.upload(u)
            lev.advance(S, 0.0, 1e-6)
            got.append(S.download())
        assert np.array_equal(got[0], got[1]), f"form {form}"
    lev.set_tiling(0)
