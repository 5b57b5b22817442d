"""What the autotuner may choose.  A refined level of 8-cell boxes in one array:
tiles over the union of the boxes fit 16x16 columns where tiles per box do not
(they would be three quarters idle), and those columns run the self-loading
form, which is the faster one."""
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [2, 4])
def test_small_boxes_in_one_array_tune_to_the_self_loading_form(order):
    from amrsolver_amd import level as L
    print(f"case autotune forms keep{order}", flush=True)
    n = (96, 96, 96)
    cls = P.closures_reference()
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    boxes = [b for b in P.decompose(n, 8) if all(b[0][d] >= 8 and b[1][d] < 88 for d in range(3)) and sum(b[0]) // 8 % 5]
    ctx = L.Context(0)
    lev = L.Level(g, boxes, cls, P.scheme(flux_euler=1, order_keep=order, visc=True), ctx=ctx)
    S = lev.new_state(layout="level")
    S.upload_ghosted(P.smooth_random_state(cls, tuple(reversed(S.tensors[0].shape[1:])), 3))
    lev.autotune(S)
    plan = lev.step_plan(S)
    print(plan, flush=True)
    assert plan["tiling"][:2] == (16, 16) and plan["tiles"] == "level" and plan["form"] == 1
