"""The tiling of a table that has not been autotuned: plane counts that fill
the workgroups a CU holds of the 8x8 kernels (viscous six, order 6 four) in
whole rounds, where cutting boxes of 8 cells shorter would only add pipeline
planes or a round; counted over the tiles that run, those of the union where
the level is one array."""
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


def _inner(n, m):
    return [b for b in P.decompose(n, m) if all(b[0][d] >= 8 and b[1][d] < n[d] - 8 for d in range(3)) and sum(b[0]) // 8 % 5]


# domain, inner boxes only, order, visc, planes a tile (8: the whole box)
CASES = {
    "800 boxes, keep6v: one round of whole boxes": ((96, 96, 96), True, 6, True, 8),
    "800 boxes, keep6": ((96, 96, 96), True, 6, False, 8),
    "800 boxes, keep4v": ((96, 96, 96), True, 4, True, 8),
    "512 boxes, keep4v: 1024 tiles, a wave each SIMD": ((64, 64, 64), False, 4, True, 4),
    "512 boxes, keep6v: 1024 tiles, one round": ((64, 64, 64), False, 6, True, 4),
}


@pytest.mark.parametrize("name", list(CASES))
def test_planes_of_8x8_columns(ctx, name):
    from amrsolver_amd import level as L
    n, inner, order, visc, planes = CASES[name]
    print(f"case default tiling {name}", flush=True)
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    lev = L.Level(g, _inner(n, 8) if inner else P.decompose(n, 8), P.closures_reference(),
                  P.scheme(flux_euler=1, order_keep=order, visc=visc), ctx=ctx)
    plan = lev.step_plan(lev.new_state(layout="boxes"))
    assert plan["tiling"][:2] == (8, 8) and min(plan["tiling"][2], 8) == planes


@pytest.mark.parametrize("order", [4, 6])
def test_planes_over_the_union(ctx, order):
    """The union's columns are far longer than its boxes of 8 cells (and far
    fewer): tiles of 64 planes would leave most of the chip idle (450 us a step
    instead of 135 at order 4)."""
    from amrsolver_amd import level as L
    n = (96, 96, 96)
    print(f"case default tiling of the union keep{order}", flush=True)
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    lev = L.Level(g, _inner(n, 8), P.closures_reference(), P.scheme(flux_euler=1, order_keep=order, visc=True), ctx=ctx)
    plan = lev.step_plan(lev.new_state(layout="level"))
    assert plan["tiles"] == "level" and plan["tiling"][:2] == (8, 8) and 4 < plan["tiling"][2] <= 10
