"""Ghost cells that a subcycled hierarchy's stages and coarse-fine
interpolation read: two coarse steps of three levels against the oracle to
1e-12 per cell (normalised per component), from smooth random states (no
symmetry plane on a box boundary, where the interpolation's limiter would
hide a wrong ghost cell), in both layouts."""
import functools
import math

import numpy as np
import pytest

from amrsolver_amd import problems as P
from conftest import rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-12
DT = 1e-4


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


def _levels():
    L = 2 * math.pi
    geoms = [P.geom((n,) * 3, (0, 0, 0), (L, L, L), (1, 1, 1)) for n in (16, 32, 64)]
    return list(zip(geoms, [P.decompose((16, 16, 16), 8),
                            [((8, 8, 4), (23, 15, 27)), ((8, 16, 4), (23, 23, 27))],
                            [((24, 24, 16), (39, 31, 47)), ((24, 32, 16), (39, 39, 47))]]))


@functools.lru_cache(maxsize=None)
def _states():
    return [P.smooth_random_state(P.closures_reference(), (n,) * 3, 31) for n in (16, 32, 64)]


def _covered(u, boxes):
    return np.concatenate([u[:, lo[2]:hi[2] + 1, lo[1]:hi[1] + 1, lo[0]:hi[0] + 1].reshape(5, -1) for lo, hi in boxes], axis=1)


@functools.lru_cache(maxsize=None)
def _oracle(order, visc):
    from oracle import oracle as O
    OH = O.OracleHierarchy(_levels())
    OH.set_state(_states())
    for k in range(2):
        OH.advance(P.closures_reference(), P.scheme(flux_euler=1, order_keep=order, visc=visc), k * DT, DT, nthreads=8)
    return [_covered(OH.get_state(lev), boxes) for lev, (_, boxes) in enumerate(_levels())]


def _run(ctx, order, visc, layout):
    from amrsolver_amd import level as L
    sch = P.scheme(flux_euler=1, order_keep=order, visc=visc)
    H = L.Hierarchy([L.Level(g, b, P.closures_reference(), sch, ctx=ctx) for g, b in _levels()], layout=layout)
    H.upload(_states())
    for k in range(2):
        H.advance(k * DT, DT)
    return [_covered(H.download(lev), boxes) for lev, (_, boxes) in enumerate(_levels())]


@pytest.mark.parametrize("layout", ["level", "boxes"])
@pytest.mark.parametrize("order,visc", [(6, True), (6, False), (4, True), (2, False)], ids=["keep6v", "keep6", "keep4v", "keep2"])
def test_hierarchy_matches_the_oracle(ctx, order, visc, layout):
    print(f"case hierarchy ghosts keep{order} visc {visc} {layout}", flush=True)
    for lev, (got, want) in enumerate(zip(_run(ctx, order, visc, layout), _oracle(order, visc))):
        err = rel_err(got, want)
        assert err <= TOL, f"level {lev}: {err:.3e}"


@pytest.mark.parametrize("order,visc", [(4, True), (2, False)], ids=["keep4v", "keep2"])
def test_hierarchy_layouts_agree(ctx, order, visc):
    """One array per box (whose stages read the other boxes' cells directly)
    and one array per level: the same bits."""
    print(f"case hierarchy layouts keep{order} visc {visc}", flush=True)
    for a, b in zip(_run(ctx, order, visc, "level"), _run(ctx, order, visc, "boxes")):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("first,second", [((0,), (-1,)), ((-1,), (0,))], ids=["fused to passes", "passes to fused"])
def test_tiling_changed_between_steps(ctx, first, second):
    """The fills follow the kernels that run: the fused stages read the other
    boxes' cells directly, the pass-structured ones read ghost cells."""
    from amrsolver_amd import level as L
    print(f"case hierarchy tiling {first} then {second}", flush=True)
    sch = P.scheme(flux_euler=1, order_keep=4, visc=True)
    H = L.Hierarchy([L.Level(g, b, P.closures_reference(), sch, ctx=ctx) for g, b in _levels()], layout="boxes")
    H.upload(_states())
    for k, tiling in enumerate((first, second)):
        H.levels[0].set_tiling(*tiling)  # the scheme's, on every level
        H.advance(k * DT, DT)
    H.levels[0].set_tiling(0)
    for lev, ((_, boxes), want) in enumerate(zip(_levels(), _oracle(4, True))):
        err = rel_err(_covered(H.download(lev), boxes), want)
        assert err <= TOL, f"level {lev}: {err:.3e}"
