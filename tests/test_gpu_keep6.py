"""The viscous KEEP order 6 stage on 16x16 columns against the same stage on
8x8 columns (another kernel, the same operations): equal to the last bit, on
tiles that end inside a box, one plane and several pieces in z, level tiles
and tiles per box, a source array, and ghost cells read from U^n; and within
1e-12 (normalised per component) of the oracle."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


def _both(lev, tz, run):
    out = []
    for t in ((8, 8, 16), (16, 16, tz)):
        lev.set_tiling(*t)
        out.append(run(t))
    lev.set_tiling(0)
    return out


@pytest.mark.parametrize("layout", ["level", "boxes"])
@pytest.mark.parametrize("n,mg,tz", [((16, 16, 4), (16, 16, 4), 4), ((17, 31, 5), (17, 31, 5), 1), ((33, 20, 9), (33, 20, 9), 4),
                                     ((15, 18, 3), (15, 18, 3), 2), ((40, 28, 6), (20, 14, 6), 6), ((48, 32, 40), (48, 32, 20), 32)])
def test_keep6_matches_other_columns(ctx, n, mg, tz, layout):
    from amrsolver_amd import level as L
    from oracle import oracle as O
    cls = P.closures_reference()
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 1, 1))
    boxes = P.decompose(n, mg)
    u = P.smooth_random_state(cls, n, 8)
    src = np.random.default_rng(4).standard_normal(u.shape) * np.max(np.abs(u), axis=(1, 2, 3))[:, None, None, None]
    for source in (None, src):
        sch = P.scheme(flux_euler=1, order_keep=6, visc=True, source=source is not None)
        lev = L.Level(g, boxes, cls, sch, ctx=ctx)
        if source is not None:
            Q = lev.new_state(ng=0)
            Q.upload(src)
            lev.set_source(Q)
        S = lev.new_state(layout=layout)

        def run(t):
            print(f"case keep6 {n} {mg} {layout} tiling {t} source {source is not None}", flush=True)
            S.upload(u)
            for _ in range(2):
                lev.advance(S, 0.0, 1e-6)
            return S.download()

        a, b = _both(lev, tz, run)
        assert np.array_equal(a, b)
        ol = O.OracleLevel(g, boxes)
        ol.set_state(u)
        for _ in range(2):
            ol.advance(cls, sch, 1e-6, source=source)
        ref = ol.get_state()
        for c in range(5):
            assert np.max(np.abs(b[c] - ref[c])) <= TOL * np.max(np.abs(ref[c]))


@pytest.mark.parametrize("tz", [16, 3])
@pytest.mark.parametrize("layout", ["level", "boxes"])
def test_keep6_refined_level(ctx, layout, tz):
    from amrsolver_amd import level as L
    g, boxes = P.tgv_amr_hierarchy(n_base=32, nlev=2)[2]
    cls = P.tgv_closures()
    lev = L.Level(g, boxes, cls, P.scheme(flux_euler=1, order_keep=6, visc=True), ctx=ctx)
    n = [g.dom_hi[d] + 1 for d in range(3)]
    full = P.tgv_state_box(cls, g, (0, 0, 0), tuple(x - 1 for x in n), 3)
    S = lev.new_state(layout=layout)

    def run(t):
        print(f"case keep6 refined {layout} tiling {t}", flush=True)
        if layout == "level":
            S.upload_ghosted(full)
        else:
            S.upload(full[:, 3:-3, 3:-3, 3:-3])
        lev.fill_patch(S)
        for _ in range(2):
            lev.advance(S, 0.0, 5e-5)
        out = np.zeros_like(full[:, 3:-3, 3:-3, 3:-3])
        got = S.download()
        for lo, hi in boxes:
            sl = (slice(None), slice(lo[2], hi[2] + 1), slice(lo[1], hi[1] + 1), slice(lo[0], hi[0] + 1))
            out[sl] = got[sl]
        return out

    a, b = _both(lev, tz, run)
    assert np.array_equal(a, b, equal_nan=True)
