"""The scalar M-step solves on the CPU against bisection in long double: branch
lengths in the default box and in boxes up to and beyond the lengths whose
expm1 overflows (the fastEM model's box [1e-6, 1000] among them), from starts
at both bounds, outside and inside; nu with branches past that length.

Tolerance 1e-12 relative: the solves end on steps whose own error is below
2e-15 x, and the objectives' slopes at the root carry a few roundings (some
4e-16 each) that a root with the slope's curvature here does not amplify by
more than 1e2."""
import numpy as np
import pytest

import mstep_reference as ref

BOXES = [(0.005, 10.0), (1e-6, 1e3), (1e-6, 705.0), (1e-3, 1e4), (1e-8, 1e6)]


def _objectives(n, seed):
    rng = np.random.default_rng(seed)
    s = np.exp(rng.uniform(np.log(1e-6), np.log(300.0), (n, 5)))
    nu = rng.choice([0.0, 1e-4, 0.3, 1.0], n) * rng.uniform(0.5, 1.0, n)
    A = (nu + 1) * s[:, 0] + nu * s[:, 1] + nu * s[:, 3]
    B = np.where(nu > 1e-5, s[:, 2] + s[:, 4], 0.0)
    return A, s[:, 1], B, nu


@pytest.mark.parametrize("dmin,dmax", BOXES)
@pytest.mark.parametrize("start", ["dmin", "dmax", "zero", "inside", "past"])
def test_branch_solve(dmin, dmax, start):
    A, S1, B, nu = _objectives(4000, 7)
    rng = np.random.default_rng(8)
    x0 = {"dmin": dmin, "dmax": dmax, "zero": 0.0, "past": 2 * dmax,
          "inside": np.exp(rng.uniform(np.log(dmin), np.log(min(dmax, 1e5)), len(A)))}[start]
    got, want = ref.branches(A, S1, B, nu, dmin, dmax, x0)
    assert ((want > dmin) & (want < dmax)).mean() > 0.5
    np.testing.assert_allclose(got, want, rtol=1e-12)


def test_branch_from_the_lower_bound_of_the_fastem_box():
    for x0 in (1e-6, 1000.0, 0.0, 0.05, 800.0):
        got, want = ref.branches([14.5], [5.0], [3.0], 0.3, 1e-6, 1e3, x0)
        assert abs(want[0] - 0.463849167) < 1e-8
        np.testing.assert_allclose(got, want, rtol=1e-12)


@pytest.mark.parametrize("spread", [0.02, 1.0])
def test_branch_solve_to_rounding(spread):
    """Warm starts in the default box: within eight roundings (2^-53 each) of the
    true root, whose slope times length is at least the objective's constant
    term (an error in either is not amplified): three in the reciprocal, two in
    the slope, one in the step, one in the result, one in the reference."""
    A, S1, B, nu = _objectives(60000, 11)
    _, want = ref.branches(A, S1, B, nu, 0.005, 10.0, 0.05)
    sel = (want > 0.005) & (want < 10.0)
    A, S1, B, nu, want = (np.ascontiguousarray(x[sel]) for x in (A, S1, B, nu, want))
    rng = np.random.default_rng(12)
    got, _ = ref.branches(A, S1, B, nu, 0.005, 10.0, want * np.exp(rng.uniform(-spread, spread, len(want))))
    np.testing.assert_allclose(got, want, rtol=8 * 2.0 ** -53)


@pytest.mark.parametrize("long_length", [0.5, 600.0, 709.0, 712.0, 1e3, 1e5])
@pytest.mark.parametrize("nu0", [0.0, 1e-6, 0.3, 0.999, 1.0])
def test_nu_solve_with_a_long_branch(long_length, nu0):
    rng = np.random.default_rng(3)
    for _ in range(40):
        n = 60
        a, b, d = rng.uniform(5, 30, n), rng.uniform(0.1, 8, n), rng.uniform(0.01, 1.0, n)
        d[0] = long_length
        a[0], b[0] = 1e-6 * rng.uniform(0.1, 2.0), rng.uniform(0.1, 8)
        got, want, evals = ref.nu_solve(a, b, d, nu0)
        assert evals > 0
        np.testing.assert_allclose(got, want, rtol=1e-12)


def test_nan_stays_nan():
    """A length or a slope that is not a number does not pass for a solution of
    nu (reported as a failed solve), and a branch falls back to its lower
    bound."""
    got, _ = ref.branches([np.nan], [1.0], [1.0], 0.5, 0.005, 10.0, 0.05)
    assert got[0] == 0.005
    _, _, evals = ref.nu_solve([1.0, 1.0], [1.0, 1.0], [np.nan, 0.1], 0.5)
    assert evals < 0
