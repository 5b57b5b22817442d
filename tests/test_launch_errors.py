"""A stage kernel that the runtime refuses to launch is reported by the stage's
launcher, for every scheme, tile and form it takes.  No GPU: a child process
puts stand-ins for the runtime's launch functions before the library's own: every
launch fails, and reading the last error clears it, as hipGetLastError does."""
import subprocess
import sys

from amrsolver_amd import capi

SHIM = """
static int last;
int __hipPushCallConfiguration(void) { return 0; }
int __hipPopCallConfiguration(void) { return 0; }
int hipLaunchKernel(void) { last = 1; return 1; }
int hipGetLastError(void) { int e = last; last = 0; return e; }
"""

CHILD = """
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
stage = getattr(lib, sys.argv[3])
class Scheme(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int32) for n in ("rhs_euler", "rhs_visc", "rhs_source", "flux_euler", "order_keep", "art_diss",
                                              "order_rk", "stages_rk")]
zeros = lambda: ctypes.create_string_buffer(4096)
for order in (2, 4, 6):
    for visc in (0, 1):
        for tx, ty in ((16, 16), (8, 8), (32, 8)):
            for form in (0, 1) if visc and order < 6 and tx == 16 else (0,):
                sch = Scheme(rhs_euler=1, rhs_visc=visc, flux_euler=1, order_keep=order, order_rk=3, stages_rk=3)
                cfg = (ctypes.c_int * 5)(tx, ty, 16, 0, form)
                rc = stage(ctypes.byref(sch), cfg, zeros(), zeros(), zeros(), None, 0, None, zeros(), zeros(), None, None,
                           None, None, zeros(), zeros())
                print(order, visc, tx, ty, form, rc)
"""


def test_refused_stage_launches_are_reported(tmp_path):
    src, shim = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(shim), str(src)], check=True)
    names = subprocess.run(["nm", "-D", "--defined-only", capi.LIBPATH], capture_output=True, text=True, check=True).stdout
    sym = [w for w in names.split() if "launch_fused_stage" in w]
    assert len(sym) == 1
    r = subprocess.run([sys.executable, "-c", CHILD, str(shim), capi.LIBPATH, sym[0]], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    rows = [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    assert len(rows) == 20
    assert [row for row in rows if row[-1] == 0] == []
