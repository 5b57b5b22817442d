"""The WENO passes' shared-reciprocal weights and their fallback: right-hand
sides bit for bit equal to the assembly of the face fluxes (whose kernel
divides as the oracle does and is held to it bit for bit) for states whose
smoothness sums lie inside, beyond and on both sides of the range the shared
reciprocal holds for."""
import numpy as np
import pytest

from amrsolver_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from amrsolver_amd import level
    return level.Context(0)


SCALES = {
    "one": lambda u: 1.0,
    "tiny, all sums below eps": lambda u: 1e-35,
    "small": lambda u: 1e-12,
    "beyond the range": lambda u: 1e9,
    "far beyond": lambda u: 1e40,
    "some lanes beyond": lambda u: np.where(np.arange(u.shape[3]) % 24 < 9, 1e9, 1.0)[None, None, None, :],
    "a flat state": lambda u: (1e3 * u[:, :1, :1, :1] / u),
}


@pytest.mark.parametrize("name", list(SCALES))
@pytest.mark.parametrize("n", [(70, 9, 5), (48, 4, 4)], ids=["box", "4x4 tube"])
def test_weno_weights_over_the_range(ctx, name, n):
    from amrsolver_amd import level as L
    print(f"case weno range {name} {n}", flush=True)
    cls = P.closures_reference()
    g = P.geom(n, (0.0, 0.0, 0.0), tuple(x / n[0] for x in n), (1, 1, 1))
    lev = L.Level(g, P.decompose(n, 64), cls, P.scheme(flux_euler=2, visc=False), ctx=ctx)
    u = P.smooth_random_state(cls, n, 5)
    u = np.ascontiguousarray(u * SCALES[name](u))
    S, D = lev.new_state(layout="boxes"), lev.new_state(layout="boxes", ng=0)
    S.upload(u)
    lev.fill_patch(S)
    F = L.FaceArrays(lev)
    lev.face_fluxes(S, F)
    lev.compute_rhs(S, D)
    rhs = D.download()
    for b, (lo, hi) in enumerate(lev.boxes):
        fx, fy, fz = (F.download(d, b) for d in range(3))
        dxi = [1.0 / g.dx[d] for d in range(3)]
        want = dxi[0] * (fx[:, :, :, :-1] - fx[:, :, :, 1:]) + dxi[1] * (fy[:, :, :-1, :] - fy[:, :, 1:, :]) + \
            dxi[2] * (fz[:, :-1, :, :] - fz[:, 1:, :, :])
        got = rhs[:, lo[2]:hi[2] + 1, lo[1]:hi[1] + 1, lo[0]:hi[0] + 1]
        assert np.isfinite(want).all()
        assert np.array_equal(got, want), f"box {b}"
    lev.close()
