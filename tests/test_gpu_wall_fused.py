"""The self-loading fused form next to bc 6 walls: steps and right-hand sides
bit for bit equal to the pass-structured kernels' (which the wall tests hold
to the oracle), on boxes whose rows end inside, at and beyond a tile, boxes
thinner than the order-reduced rows, and one box between both walls."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


def _rows(n, edges):
    """Boxes cut along y at `edges` (and in x at 16)."""
    ys = [0] + list(edges) + [n[1]]
    return [((x0, y0, 0), (min(x0 + 16, n[0]) - 1, y1 - 1, n[2] - 1))
            for y0, y1 in zip(ys, ys[1:]) for x0 in range(0, n[0], 16)]


CASES = {
    "one box, 20 rows": ((32, 20, 9), ()),
    "16 and 9 rows": ((33, 25, 6), (16,)),
    "8, 16 and 15 rows": ((16, 39, 5), (8, 24)),
    "9 rows to each wall": ((32, 18, 7), (9,)),
    "walls 2 rows and 1 row deep": ((16, 35, 4), (2, 18, 34)),
    "32 rows, tiles end at the walls": ((16, 32, 17), ()),
}


@pytest.mark.parametrize("layout", ["level", "boxes"])
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("order,body", [(4, True), (4, False), (2, True)], ids=["keep4 body", "keep4", "keep2 body"])
def test_wall_rows_match_the_passes(ctx, name, layout, order, body):
    from amrsolver_amd import level as L
    n, edges = CASES[name]
    print(f"case wall fused {name} {layout} keep{order} body {body}", flush=True)
    cls, g, _, parm = P.wall_channel(n)
    sch = P.scheme(flux_euler=1, order_keep=order, visc=True, order_rk=3, stages_rk=3, source=body)
    lev = L.Level(g, _rows(n, edges), cls, sch, ctx=ctx)
    lev.set_problem(wall_T=parm["Tw"], body_force_x=parm["fx"] if body else 0.0)
    rng = np.random.default_rng(7)
    u = P.wall_channel_state(cls, g, n, parm)
    u[3] = u[0] * 30.0 * rng.uniform(-1, 1, size=u.shape[1:])  # w, so that every component varies
    u[4] += 0.5 * u[3] ** 2 / u[0]
    out = []
    S, D = lev.new_state(layout=layout), lev.new_state(layout=layout, ng=0)
    for passes in (True, False):
        if passes:
            lev.set_tiling(-1)
        plan = lev.step_plan(S)
        assert plan["tiles"] == ("passes" if passes else "boxes")
        assert passes or plan["form"] == 1
        S.upload(u)
        lev.fill_patch(S)
        lev.compute_rhs(S, D)
        for _ in range(2):
            lev.advance(S, 0.0, 2e-9)
        out.append((D.download(), S.download()))
        lev.set_tiling(0)
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])
    assert np.isfinite(out[1][1]).all()
    lev.close()
