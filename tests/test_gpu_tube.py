"""Stages of 1D problems in one kernel (boxes 4 x 4 cells across, periodic in
y and z): steps bit for bit equal to the directional passes' on the same
problem repeated once in y (8 cells across, which the one-kernel stages do not
take), for short and long bricks (few and many cells), brick ends and
remainders, every kind of x side, sources and batches with their own steps."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


def _geom(L, ny, per=False, lo=2, hi=2):
    g = P.geom((L, ny, 4), (0.0, 0.0, 0.0), (1.0, ny / L, 4 / L), (int(per), 1, 1), lo_bc=(lo, 0, 0), hi_bc=(hi, 0, 0))
    for d in range(3):
        g.dx[d] = 1.0 / L
    return g


def _state(cls, L, seed):
    u = P.smooth_random_state(cls, (L, 4, 4), seed, ampl=0.2, u0=60.0)
    u[0, :, :, L // 2:] *= 0.4  # a jump
    return u


# x cuts, periodic x, bc codes; the first four are few cells (split bricks)
LEVELS = {
    "3, 4 and 5 cells": ((3, 7, 12), False, 2, 2),
    "one periodic box of 17": ((17,), True, 0, 0),
    "periodic, 46 cells in 3 boxes": ((15, 31, 46), True, 0, 0),
    "reflecting, 64 and 7 cells": ((64, 71), False, 3, 4),
    "long bricks, 16, 1600 and 15 cells": ((16, 1616, 1631), False, 2, 3),
    "long bricks, one periodic box": ((1700,), True, 0, 0),
}


@pytest.mark.parametrize("flux", [2, 0], ids=["weno", "muscl"])
@pytest.mark.parametrize("name", list(LEVELS))
@pytest.mark.parametrize("rk,src", [((3, 3), False), ((3, 4), True), ((2, 3), False)], ids=["rk33", "rk34 src", "rk23"])
def test_tube_levels_match_the_passes(ctx, name, flux, rk, src):
    from amrsolver_amd import level as L
    print(f"case tube {name} flux {flux} rk {rk} src {src}", flush=True)
    cuts, per, lo, hi = LEVELS[name]
    n = cuts[-1]
    cls = P.closures_reference()
    u = _state(cls, n, 11)
    q = np.random.default_rng(3).standard_normal(u.shape) * np.max(np.abs(u), axis=(1, 2, 3))[:, None, None, None]
    sch = P.scheme(flux_euler=flux, visc=False, order_rk=rk[0], stages_rk=rk[1], source=src)
    out = []
    for rep in (1, 2):
        g = _geom(n, 4 * rep, per, lo, hi)
        boxes = [((a, 0, 0), (b - 1, 4 * rep - 1, 3)) for a, b in zip((0,) + cuts[:-1], cuts)]
        lev = L.Level(g, boxes, cls, sch, ctx=ctx)
        if src:
            Q = lev.new_state(layout="boxes", ng=0)
            Q.upload(np.tile(q, (1, 1, rep, 1)))
            lev.set_source(Q)
            lev.set_problem(body_force_x=0.3)
        S = lev.new_state(layout="boxes")
        S.upload(np.tile(u, (1, 1, rep, 1)))
        lev.clock_set(0.0)
        lev.advance_cfl(S, 0.3, -1.0, 2)
        lev.advance(S, 0.0, 1e-7)
        out.append(S.download())
        lev.close()
    assert np.isfinite(out[0]).all()
    assert np.array_equal(out[0], out[1][:, :, :4]) and np.array_equal(out[0], out[1][:, :, 4:])


@pytest.mark.parametrize("flux", [2, 0], ids=["weno", "muscl"])
@pytest.mark.parametrize("lengths", [(3, 16, 61, 64, 90), (700, 15, 512, 31, 450, 3)], ids=["short bricks", "long bricks"])
def test_tube_batches_match_the_passes(ctx, flux, lengths):
    from amrsolver_amd import level as L
    print(f"case tube batch {lengths} flux {flux}", flush=True)
    cls = P.closures_reference()
    sch = P.scheme(flux_euler=flux, visc=False)
    out = []
    for rep in (1, 2):
        bat = L.Batch([_geom(n, 4 * rep) for n in lengths], cls, sch, ctx=ctx)
        S = bat.new_state()
        S.upload_problems([np.tile(_state(cls, n, k), (1, 1, rep, 1)) for k, n in enumerate(lengths)])
        dts = bat.est_time_steps(S, 0.3)
        dts[1] = 0.0  # a finished problem is left untouched
        for _ in range(2):
            bat.advance_dt(S, dts)
        bat.clock_set(0.0)
        bat.advance_cfl(S, 0.3, 1e-3, 2)
        out.append(S.download_problems())
        bat.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b[:, :, :4]) and np.array_equal(a, b[:, :, 4:])
