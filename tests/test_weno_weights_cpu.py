"""The WENO weights that share one reciprocal (weno5js_fast) against the plain
form, compiled for the CPU from the same header: the fast form holds, and gives
the plain form's bits, for stencils whose values differ by up to 1e18 (flux
differences of strong detonations in CGS units are some 1e15), flat parts and
single jumps among them; beyond, and for NaN and infinities, it says that it
does not hold, or differs by less than the values' own rounding.  The GPU's reciprocal instruction is stood in for by one of 23
bits, so the refinement has its work to do."""
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
static inline double rcp23(double d) {
  double r = 1.0 / d;
  uint64_t b;
  memcpy(&b, &r, 8);
  b &= ~((uint64_t(1) << 29) - 1);
  memcpy(&r, &b, 8);
  return r;
}
#define __builtin_amdgcn_rcp rcp23
#include "cns_point.h"
int main() {
  std::mt19937_64 g(20261205);
  std::uniform_real_distribution<double> u(-1, 1), e(-30, 18);
  long refused = 0, differ = 0, n = 0;
  for (int k = 0; k < 2000000; ++k) {
    const double sc = std::pow(10.0, k % 4 ? e(g) : 18.0 - 0.5 * (k % 9));
    double s[5];
    const int kind = k % 5;
    for (int i = 0; i < 5; ++i) {
      s[i] = sc * u(g);
      if (kind == 1) s[i] = sc * (1.0 + 1e-6 * i);                 // nearly linear
      if (kind == 2) s[i] = i <= k % 4 ? sc : 0.25 * sc;           // one jump between flat parts
      if (kind == 3) s[i] = sc * (i <= k % 4 ? 1.0 : 1e-9 * u(g));  // a jump into a nearly flat part
    }
    bool ok = true;
    const double a = amr::weno5js_fast(s[0], s[1], s[2], s[3], s[4], ok);
    const double b = amr::weno5js(s[0], s[1], s[2], s[3], s[4]);
    ++n;
    if (!ok) ++refused;
    else if (memcmp(&a, &b, 8)) ++differ;
  }
  // far outside: refused, or no further from the plain form than 8 roundings
  // of the largest value
  long wrong = 0;
  const double out[] = {1e19, 1e20, 1e30, 1e37, 1e38, 1e39, 1e60, 1e75, 1e76, 1e77, 1e80, 1e160, 1e300, INFINITY, NAN};
  for (double x : out)
    for (int at = 0; at < 5; ++at)
      for (int to = at; to < 5; ++to)
        for (double rest : {0.0, 1.0, 1e5}) {
          double s[5];
          for (int i = 0; i < 5; ++i) s[i] = i >= at && i <= to ? x : rest;
          bool ok = true;
          const double a = amr::weno5js_fast(s[0], s[1], s[2], s[3], s[4], ok);
          const double b = amr::weno5js(s[0], s[1], s[2], s[3], s[4]);
          if (ok && memcmp(&a, &b, 8) && !(std::fabs(a - b) <= 8 * 0x1p-53 * x)) ++wrong;
        }
  std::printf("%ld %ld %ld %ld\n", n, refused, differ, wrong);
  return 0;
}
"""

STUB = """
#pragma once
#define __host__
#define __device__
#define __forceinline__ inline
"""


@pytest.fixture(scope="module")
def counts(tmp_path_factory):
    d = tmp_path_factory.mktemp("weno")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(STUB)
    (d / "t.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-I", str(d), "-I", f"{ROOT}/include", "-I",
                    f"{ROOT}/amrsolver_amd/csrc", "-o", str(d / "t"), str(d / "t.cpp")], check=True)
    r = subprocess.run([str(d / "t")], capture_output=True, text=True, check=True)
    return dict(zip(("n", "refused", "differ", "wrong"), map(int, r.stdout.split())))


def test_the_fast_form_holds_over_its_range(counts):
    assert counts["n"] == 2000000 and counts["refused"] == 0


def test_the_fast_form_has_the_plain_forms_bits(counts):
    assert counts["differ"] == 0


def test_the_fast_form_is_refused_or_harmless_outside(counts):
    assert counts["wrong"] == 0
