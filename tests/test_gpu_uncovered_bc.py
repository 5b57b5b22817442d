"""Levels that cover part of a bounded domain: a boundary's ghost cells take
their values from cells of the stage input, also from ghost cells no box covers
(which keep the caller's values of U^n through a step).  Fused steps bit for bit
against the pass-structured kernels', which copy those cells into every stage
input, after a step of theirs from another state has left that state's values in
the stage workspaces."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


# periodic directions, boundary codes lo and hi
BCS = {
    "z slip and symmetry": ((1, 1, 0), (0, 0, 4), (0, 0, 3)),
    "y and z bounded": ((1, 0, 0), (0, 2, 3), (0, 3, 3)),
    "x outflow": ((0, 1, 1), (2, 0, 0), (2, 0, 0)),
}
BOXES = {
    "8 cells deep": ((24, 24, 32), 8),
    "16 and 8 cells": ((40, 24, 48), 16),
}


def _upload(S, lev, n, cls, seed):
    full = P.smooth_random_state(cls, tuple(m + 6 for m in n), seed)
    if S.layout == "level":
        S.upload_ghosted(full)
    else:
        for b, (lo, hi) in enumerate(lev.boxes):
            S.upload_box(b, full[:, lo[2]:hi[2] + 7, lo[1]:hi[1] + 7, lo[0]:hi[0] + 7])


@pytest.mark.parametrize("layout", ["level", "boxes"])
@pytest.mark.parametrize("order", [2, 4, 6])
@pytest.mark.parametrize("cut", list(BOXES))
@pytest.mark.parametrize("bc", list(BCS))
def test_boundaries_beside_uncovered_cells(ctx, bc, cut, order, layout):
    from amrsolver_amd import level as L
    print(f"case uncovered bc {bc} {cut} keep{order} {layout}", flush=True)
    n, mg = BOXES[cut]
    cls = P.closures_reference()
    per, lo, hi = BCS[bc]
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), per, lo_bc=lo, hi_bc=hi)
    boxes = [b for k, b in enumerate(P.decompose(n, mg)) if k % 3 != 1]
    lev = L.Level(g, boxes, cls, P.scheme(flux_euler=1, order_keep=order, visc=True), ctx=ctx)
    out = []
    for tiling in (-1, 0):
        lev.set_tiling(-1)
        S = lev.new_state(layout=layout)
        _upload(S, lev, n, cls, 5)
        lev.advance(S, 0.0, 1e-6)
        lev.set_tiling(tiling)
        _upload(S, lev, n, cls, 6)
        for _ in range(2):
            lev.advance(S, 0.0, 1e-6)
        u = S.download()
        out.append([u[:, l[2]:h[2] + 1, l[1]:h[1] + 1, l[0]:h[0] + 1] for l, h in boxes])
    lev.set_tiling(0)
    assert all(np.isfinite(a).all() for a in out[1])
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    lev.close()


def test_levels_away_from_boundaries_read_from_un(ctx):
    """No copy pass where no boundary lies beside uncovered cells."""
    from amrsolver_amd import level as L
    n = (48, 48, 48)
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 0, 0), lo_bc=(0, 2, 4), hi_bc=(0, 2, 4))
    boxes = [((16, 16, 16), (31, 31, 31))]
    lev = L.Level(g, boxes, P.closures_reference(), P.scheme(flux_euler=1, order_keep=4, visc=True), ctx=ctx)
    assert lev.step_plan(lev.new_state(layout="level"))["uncovered_from_un"]
