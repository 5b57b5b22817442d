"""Level tiles of boxes whose bounding box has corners no box covers: they read
only what the arrays and workspaces hold (a stage input's array spans its boxes'
windows, grown by three cells), and give the pass-structured kernels' bits.  On
the CPU with kernels and host code compiled for it and every allocation against
pages that fault."""
import os
import platform
import subprocess
import sys

import numpy as np
import pytest

import cpu_hip
from amrsolver_amd import problems as P
from conftest import ROOT

# a low box and a high one beside each other in y, next to a symmetry boundary
# (so that the stages read every cell from their inputs): below and above the
# windows' planes lie columns of the bounding box that hold nothing
LEVELS = {
    "low behind": ((16, 28, 40), [((0, 0, 16), (15, 3, 23)), ((0, 8, 8), (15, 11, 15))]),
    "low in front": ((16, 28, 40), [((0, 0, 8), (15, 3, 15)), ((0, 8, 16), (15, 11, 23))]),
}
SCHEMES = {"keep4 visc": (4, True), "keep6 visc": (6, True), "keep6": (6, False)}


def check(L, name, scheme, source):
    n, boxes = LEVELS[name]
    order, visc = SCHEMES[scheme]
    cls = P.closures_reference()
    g = P.geom(n, (0.0, 0.0, 0.0), (1.0, 0.8, 0.7), (1, 0, 1), lo_bc=(0, 3, 0), hi_bc=(0, 3, 0))
    lev = L.Level(g, boxes, cls, P.scheme(flux_euler=1, order_keep=order, visc=visc, source=source), ctx=L.Context(0))
    if source:
        Q = lev.new_state(layout="level")
        Q.upload(np.random.default_rng(4).standard_normal((5, *n[::-1])))
        lev.set_source(Q)
    out = []
    for tiling in ((-1, 0, 0), (16, 16, 8), (8, 8, 6), (32, 8, 16)):
        lev.set_tiling(*tiling)
        S = lev.new_state(layout="level")
        S.upload_ghosted(P.smooth_random_state(cls, tuple(m + 6 for m in n), 3))
        plan = lev.step_plan(S)
        assert plan["tiles"] == ("passes" if tiling[0] == -1 else "level"), plan
        for _ in range(2):
            lev.advance(S, 0.0, 1e-6)
        u = S.download()
        out.append([u[:, l[2]:h[2] + 1, l[1]:h[1] + 1, l[0]:h[0] + 1] for l, h in boxes])
    assert all(np.isfinite(a).all() for a in out[0])
    for got in out[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(out[0], got))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if platform.machine() != "x86_64" or not os.path.exists(cpu_hip.CLANG):
        pytest.skip("fibers for x86-64, ROCm's clang")
    return cpu_hip.build(str(tmp_path_factory.mktemp("cpu")))


@pytest.mark.parametrize("front", [False, True], ids=["ends guarded", "fronts guarded"])
@pytest.mark.parametrize("scheme", list(SCHEMES))
@pytest.mark.parametrize("name", list(LEVELS))
def test_loads_stay_in_the_arrays(lib, name, scheme, front):
    code = (f"import sys; sys.path[:0] = [{ROOT!r}, {os.path.dirname(__file__)!r}]\n"
            f"import cpu_hip, test_level_edges as t\nL = cpu_hip.use({lib!r})\n"
            f"for source in (False, True): t.check(L, {name!r}, {scheme!r}, source)")
    env = dict(os.environ, CPU_HIP_FRONT="1") if front else None
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]


@pytest.mark.gpu
@pytest.mark.parametrize("source", [False, True], ids=["", "source"])
@pytest.mark.parametrize("scheme", list(SCHEMES))
@pytest.mark.parametrize("name", list(LEVELS))
def test_steps_match_the_passes(name, scheme, source):
    from amrsolver_amd import level
    print(f"case level edges {name} {scheme} source {source}", flush=True)
    check(level, name, scheme, source)
