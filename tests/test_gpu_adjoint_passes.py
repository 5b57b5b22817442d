"""Gradients of runs whose forward stages are the pass-structured kernels' on a
periodic level held in one array (asked for, or taken for boxes that leave the
tiles' lanes idle): those kernels read the ghost cells of every stage input,
which therefore have to be filled.  Against the same run with one array per box:
the two reverse sweeps differ in association only, to 1e-12 a stage
(test_gpu_adjoint_march's bar), six stages."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu

LEVELS = {"asked for": ((24, 20, 16), (12, 10, 16), -1), "narrow boxes": ((12, 16, 24), (4, 4, 6), 0)}


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


@pytest.mark.parametrize("order,visc", [(2, True), (4, True), (6, False)], ids=["keep2v", "keep4v", "keep6"])
@pytest.mark.parametrize("name", list(LEVELS))
def test_gradient_of_one_array_equals_boxes(ctx, name, order, visc):
    from amrsolver_amd import level as L
    print(f"case adjoint passes {name} keep{order}", flush=True)
    n, mg, tiling = LEVELS[name]
    cls = P.closures_scaled_sutherland(0.02, T0=300.0)
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    lev = L.Level(g, P.decompose(n, mg), cls, P.scheme(flux_euler=1, order_keep=order, visc=visc), ctx=ctx)
    lev.set_tiling(tiling)
    u = P.smooth_random_state(cls, n, 5)
    got = {}
    for layout in ("boxes", "level"):
        S, G = lev.new_state(layout=layout), lev.new_state(layout=layout, ng=0)
        S.upload(u)
        J = lev.adjoint_run(S, 1e-5, 2, 1, G)
        got[layout] = (J, G.download())
    lev.set_tiling(0)
    lev.close()
    (Jb, gb), (Jl, gl) = got["boxes"], got["level"]
    assert np.isfinite(gb).all()
    assert abs(Jl - Jb) <= 1e-13 * abs(Jb)
    for k in range(5):
        assert np.max(np.abs(gl[k] - gb[k])) <= 6e-12 * np.max(np.abs(gb[k])), f"component {k}"
