"""The engine's scalar M-step solves (laml_amd/csrc/pmm_solve.hpp) built for the
host, next to reference solutions by bisection in long double on the same
objectives (EM_solver.py:349-407): argmax of a branch's objective over a box,
argmax of the nu objective over [0, 1]."""
import ctypes
import os
import subprocess
import tempfile

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_f64 = np.ctypeslib.ndpointer(dtype=np.float64, flags="C")
_i32 = np.ctypeslib.ndpointer(dtype=np.int32, flags="C")

SOURCE = r"""
#include <math.h>
#include <string.h>
#include <stdint.h>
#define __device__
#define __forceinline__ inline
// the hardware's estimate is good to some 24 bits
static inline double rcp_estimate(double x) {
  double r = 1.0 / x;
  uint64_t u;
  memcpy(&u, &r, 8);
  u &= ~((uint64_t)0x0fffffff);
  memcpy(&r, &u, 8);
  return r;
}
#define __builtin_amdgcn_rcp rcp_estimate
#include "pmm_solve.hpp"
using namespace laml;
typedef long double LD;
static LD slope(const BranchObj& o, LD d) {
  return o.S1 / expm1l(d) + (o.B > 0.0 ? o.B * (LD)o.nu / expm1l((LD)o.nu * d) : 0.0L) - o.A;
}
extern "C" {
void branches(int n, const double* A, const double* S1, const double* B, const double* nu, double dmin, double dmax,
              const double* x0, double* got, double* want) {
  for (int i = 0; i < n; ++i) {
    const BranchObj o{A[i], S1[i], B[i], nu[i]};
    got[i] = solve_branch(o, dmin, dmax, x0[i]);
    LD lo = dmin, hi = dmax;
    if (!(slope(o, lo) > 0)) { want[i] = dmin; continue; }
    if (!(slope(o, hi) < 0)) { want[i] = dmax; continue; }
    for (int k = 0; k < 120; ++k) {
      const LD m = 0.5L * (lo + hi);
      if (slope(o, m) > 0) lo = m; else hi = m;
    }
    want[i] = (double)lo;
  }
}
// returns the evaluations the solve took (negative: not converged)
int nu_solve(int n, const double* a, const double* b, const double* d, double nu0, double* got, double* want) {
  double x = nu_start(nu0), lo = 0.0, hi = 2.0, xn = x;
  bool fin = false;
  int e = 0;
  for (; e < 200 && !fin; ++e) {
    NuSum s{0.0, 0.0, 0.0, 0.0};
    for (int i = 0; i < n; ++i) nu_term(a[i], b[i], d[i], x, s);
    fin = nu_step(x, s, lo, hi, xn);
    x = xn;
  }
  *got = x;
  auto g = [&](LD y) {
    LD s = 0;
    for (int i = 0; i < n; ++i)
      if (b[i] != 0.0) s += (LD)d[i] * (b[i] / expm1l(y * d[i]) - a[i]);
    return s;
  };
  LD l = 0, h = 1;
  if (g(1) > 0) l = 1;
  for (int k = 0; k < 200 && l < 1; ++k) {
    const LD m = 0.5L * (l + h);
    if (g(m) > 0) l = m; else h = m;
  }
  *want = (double)l;
  return fin ? e : -e;
}
}
"""

_lib = None


def lib():
    global _lib
    if _lib is None:
        with tempfile.TemporaryDirectory() as tmp:
            src, so = os.path.join(tmp, "solve.cpp"), os.path.join(tmp, "solve.so")
            with open(src, "w") as f:
                f.write(SOURCE)
            subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I",
                            os.path.join(ROOT, "laml_amd", "csrc"), src, "-o", so, "-lm"], check=True)
            L = ctypes.CDLL(so)
        D = ctypes.c_double
        L.branches.argtypes = [ctypes.c_int, _f64, _f64, _f64, _f64, D, D, _f64, _f64, _f64]
        L.branches.restype = None
        L.nu_solve.argtypes = [ctypes.c_int, _f64, _f64, _f64, D, _f64, _f64]
        _lib = L
    return _lib


def _vec(x, n):
    return np.ascontiguousarray(np.broadcast_to(np.asarray(x, dtype=np.float64), (n,)))


def branches(A, S1, B, nu, dmin, dmax, x0):
    """(engine's, reference's) branch lengths of the objectives."""
    n = len(A)
    got, want = np.empty(n), np.empty(n)
    lib().branches(n, _vec(A, n), _vec(S1, n), _vec(B, n), _vec(nu, n), dmin, dmax, _vec(x0, n), got, want)
    return got, want


def nu_solve(a, b, d, nu0):
    """(engine's nu, reference's nu, evaluations; negative: not converged)."""
    n = len(a)
    got, want = np.empty(1), np.empty(1)
    e = lib().nu_solve(n, _vec(a, n), _vec(b, n), _vec(d, n), nu0, got, want)
    return got[0], want[0], e


def mstep(counts, K, nu0, dmin, dmax):
    """Reference M-step of a problem whose branches are all free, on raw
    counts [N, 5] over K sites: (branch lengths, nu)."""
    s = np.maximum(1e-6, np.asarray(counts, dtype=np.float64))
    s = s / s.sum(1, keepdims=True) * K
    A = (nu0 + 1) * s[:, 0] + nu0 * s[:, 1] + nu0 * s[:, 3]
    B = s[:, 2] + s[:, 4] if nu0 > 1e-5 else np.zeros(len(s))
    _, d = branches(A, s[:, 1], B, nu0, dmin, dmax, 0.5 * (dmin + dmax))
    _, nu, _ = nu_solve(s[:, 0] + s[:, 1] + s[:, 3], s[:, 2] + s[:, 4], d, 0.5)
    return d, nu
