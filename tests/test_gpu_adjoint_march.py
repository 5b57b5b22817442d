"""The marching reverse stage (periodic level in one array, KEEP order 2/4)
against the pass-structured reverse of the same stage (one array per box): the
edges of its 16x16 tiles, one plane and several pieces in z, boxes meeting
inside a tile row, both orders, with and without viscosity, the three stage
combinations, lam_s1 apart from, and the same as, lam_sin.

Both gather the same few hundred products per cell in FP64 and differ in
association only: a cell's sum is off by at most some 300 * 2^-53 = 3e-14 of
its absolute terms, whose sum stays within 30 times the largest entry of a
component on these states; the bar is 1e-12 of that entry."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu

SIZES = [((16, 16, 4), (16, 16, 4)), ((17, 31, 5), (17, 31, 5)), ((33, 30, 9), (33, 30, 9)), ((14, 15, 21), (14, 15, 21)),
         ((48, 32, 20), (32, 16, 12)), ((40, 28, 6), (20, 14, 6)), ((12, 13, 3), (12, 13, 3)), ((96, 80, 33), (48, 80, 33))]
STAGES = [(0, (0.75, 0.25, 1.0, 2e-2)), (1, (0.5, 0.0, 0.7, 3e-2)), (2, (0.0, 0.0, 0.0, 0.0))]


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("visc", [True, False], ids=["visc", "euler"])
@pytest.mark.parametrize("n,mg", SIZES, ids=["x".join(map(str, s[0])) for s in SIZES])
def test_march_matches_passes(ctx, n, mg, visc, order):
    from amrsolver_amd import level as L
    cls = P.closures_scaled_sutherland(0.02, T0=300.0)
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    sch = P.scheme(flux_euler=1, order_keep=order, visc=visc)
    lev = L.Level(g, P.decompose(n, mg), cls, sch, ctx=ctx)
    u = P.smooth_random_state(cls, n, 5)
    rng = np.random.default_rng(17)
    lam, s0, s1 = (rng.standard_normal(u.shape) for _ in range(3))
    for mode, coef in STAGES:
        for shared in (False, True):
            for acc in (False, True):
                print(f"case march {n} {mg} visc {visc} order {order} mode {mode} shared {shared} acc {acc}", flush=True)
                got = {}
                for layout in ("level", "boxes"):
                    S = lev.new_state(layout=layout)
                    Lo, Li, L1 = (lev.new_state(layout=layout, ng=0) for _ in range(3))
                    S.upload(u)
                    lev.fill_patch(S)
                    Lo.upload(lam)
                    Li.upload(s0)
                    L1.upload(s1)
                    lev.vjp_stage(mode, *coef, S, Lo, Li if shared else L1, Li, accumulate=acc)
                    got[layout] = (Li.download(), L1.download())
                for a, b in zip(got["level"], got["boxes"]):
                    for k in range(5):
                        assert np.max(np.abs(a[k] - b[k])) <= 1e-12 * np.max(np.abs(b[k])), f"component {k}"


def test_march_with_outputs_per_box(ctx):
    """State and stage adjoint in one array, the arrays that receive the result
    one per box: the same bits as with all in one array."""
    from amrsolver_amd import level as L
    n, mg = (48, 32, 20), (32, 16, 12)
    cls = P.closures_scaled_sutherland(0.02, T0=300.0)
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    lev = L.Level(g, P.decompose(n, mg), cls, P.scheme(flux_euler=1, order_keep=4, visc=True), ctx=ctx)
    u = P.smooth_random_state(cls, n, 5)
    rng = np.random.default_rng(18)
    lam, s0, s1 = (rng.standard_normal(u.shape) for _ in range(3))
    S, Lo = lev.new_state(), lev.new_state(ng=0)
    S.upload(u)
    lev.fill_patch(S)
    Lo.upload(lam)
    got = []
    for layout in ("level", "boxes"):
        print(f"case march outputs {layout}", flush=True)
        Li, L1 = (lev.new_state(layout=layout, ng=0) for _ in range(2))
        Li.upload(s0)
        L1.upload(s1)
        lev.vjp_stage(0, 0.75, 0.25, 1.0, 2e-2, S, Lo, L1, Li, accumulate=True)
        got.append((Li.download(), L1.download()))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
