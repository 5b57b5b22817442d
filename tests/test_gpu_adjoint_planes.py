"""The marching reverse stage on tiles of several planes, whose sums run over
three planes at once: against the pass-structured reverse of the same stage
(one array per box), at sizes for which tiles of 3, 4, 7, 11 and 14 planes are
estimated fastest (orders 4 and viscous 2; inviscid order 2 takes 2 to 10),
with a shorter last piece in z.  The bar is test_gpu_adjoint_march's, for its
reason: the two differ in association only."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu

SIZES = [((110, 94, 29), (55, 94, 29)), ((128, 64, 64), (64, 64, 64)), ((96, 96, 96), (96, 96, 48)),
         ((130, 126, 64), (65, 63, 64)), ((200, 180, 37), (100, 90, 37))]
STAGES = [(0, (0.75, 0.25, 1.0, 2e-2), False, True), (1, (0.5, 0.0, 0.7, 3e-2), True, False), (2, (0.0, 0.0, 0.0, 0.0), False, False)]


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


@pytest.mark.parametrize("order,visc", [(4, True), (2, True), (4, False), (2, False)], ids=["keep4v", "keep2v", "keep4", "keep2"])
@pytest.mark.parametrize("n,mg", SIZES, ids=["3 planes", "4 planes", "7 planes", "11 planes", "14 planes"])
def test_march_of_several_planes_matches_passes(ctx, n, mg, order, visc):
    from amrsolver_amd import level as L
    cls = P.closures_scaled_sutherland(0.02, T0=300.0)
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    lev = L.Level(g, P.decompose(n, mg), cls, P.scheme(flux_euler=1, order_keep=order, visc=visc), ctx=ctx)
    u = P.smooth_random_state(cls, n, 5)
    rng = np.random.default_rng(19)
    lam, s0, s1 = (rng.standard_normal(u.shape) for _ in range(3))
    for mode, coef, shared, acc in STAGES:
        print(f"case march planes {n} {mg} visc {visc} order {order} mode {mode} shared {shared} acc {acc}", flush=True)
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
    lev.close()
