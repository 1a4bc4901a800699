"""The FP64 Boys lookup of the shell-pair ERI engine (csrc/boys_fp64.h), compiled
for the host: at the end of its table it stays on the table's rows (a row of NaN
lies behind them) and gives F_m there too.  Tolerance: the first term left out
is 0.1^10 / 10! / 31 = 9e-19; ten to twenty roundings of values up to 1 in the
lookup and as many in the incomplete gamma function: 1e-14."""
import os
import subprocess

import numpy as np
import pytest
from scipy import special

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "pyscf_ipu_amd", "csrc", "boys_fp64.h")
EDGE = 39.9
MAIN = r"""
#define __device__
#define __forceinline__ inline
#include "%s"
#include <stdio.h>
using namespace pscf;
static double tab[(BOYSD_NT + 1) * BOYSD_COLS], f[8];
template <int L> void run(double t) { ep_boys<L>(t, tab, f); }
int main() {
  int L;
  double t;
  scanf("%%d", &L);
  for (int i = 0; i < BOYSD_NT * BOYSD_COLS; ++i) scanf("%%lf", tab + i);
  for (int k = 0; k < BOYSD_COLS; ++k) tab[BOYSD_NT * BOYSD_COLS + k] = NAN;
  while (scanf("%%lf", &t) == 1) {
    switch (L) {
      case 0: run<0>(t); break;
      case 2: run<2>(t); break;
      default: run<5>(t); break;
    }
    for (int m = 0; m <= L; ++m) printf("%%.17g ", f[m]);
    printf("\n");
  }
}
"""


def _boys(m, t):
    t = np.asarray(t, dtype=np.float64)
    a, x = m + 0.5, np.maximum(t, 1e-20)
    return np.where(t == 0, 1 / (2 * m + 1), special.gammainc(a, x) * special.gamma(a) / (2 * x ** a))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("boys")
    src, exe = d / "boys.cpp", d / "boys"
    src.write_text(MAIN % HEADER)
    subprocess.run(["g++", "-O1", "-std=c++17", str(src), "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("L", [0, 2, 5])
def test_fp64_lookup_ends_with_its_table(program, L):
    nodes = 0.2 * np.arange(200)
    fact = [special.factorial(k) for k in range(11)]
    tab = np.stack([_boys(L + k, nodes) / fact[k] for k in range(11)] + [np.exp(-nodes)], 1)
    below = [np.nextafter(EDGE, 0), EDGE, 39.85, 39.7, 39.6999, 0.0, 0.1, 0.0999]
    above = [np.nextafter(EDGE, 99), 40.0, 1e4, 1e300, np.inf]  # clamped; the caller takes the asymptote
    text = " ".join(repr(float(x)) for x in [*tab.ravel(), *below, *above])
    out = subprocess.run([program], input=f"{L} {text}", capture_output=True, text=True, check=True).stdout
    got = np.array([[float(x) for x in line.split()] for line in out.splitlines()])
    assert got.shape == (len(below) + len(above), L + 1)
    ref = np.stack([_boys(m, np.minimum(below + above, EDGE)) for m in range(L + 1)], 1)
    assert np.isfinite(got).all() and np.abs(got - ref).max() < 1e-14
