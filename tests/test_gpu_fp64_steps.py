"""The FP64-exact tracers' rules for their short sequences: each case sits on
one side of a rule, and the vertices (or counts) must be the oracle's bit for
bit on either."""
import numpy as np
import pytest

import oracle as O
from onekapy_amd import Realizations, trace_vertices

pytestmark = pytest.mark.gpu

COEF = (1e-5, -2e-5, 0.0, 1e-2, -5e-3, 2000.0)
# wells (x, y, r, q), start point, coefficients A..F, porosity, thickness
RULES = {
    # no zero coordinate: only the points' upper bound is checked
    "all_nonzero": ([(500.0, 300.0, 0.25, 700.0), (900.0, 650.0, 0.25, 400.0)],
                    (501.25, 300.0), COEF, 0.25, 20.0),
    # a well and the origin on the axes: points pass the lower bound too,
    # the first one with a coordinate of exactly 0
    "zero_well_coordinate": ([(0.0, 0.0, 0.25, 700.0), (0.0, 650.0, 0.25, 400.0)],
                             (0.0, -1.25), COEF, 0.25, 20.0),
    "subnormal_start": ([(0.0, 0.0, 0.25, 700.0), (300.0, 650.0, 0.25, 400.0)],
                        (1.0e-310, 1.25), COEF, 0.25, 20.0),
    # a regional coefficient below 2^-200, and one above 2^100
    "tiny_coefficient": ([(500.0, 300.0, 0.25, 700.0)], (501.25, 300.0),
                         (1e-5, -2e-5, 1e-70, 1e-2, -5e-3, 2000.0), 0.25, 20.0),
    "huge_coefficient": ([(500.0, 300.0, 0.25, 700.0)], (501.25, 300.0),
                         (1e-5, -2e-5, 0.0, 2e30, -5e-3, 2000.0), 0.25, 20.0),
    # thickness x porosity below 2^-100
    "tiny_bn": ([(500.0, 300.0, 0.25, 7e-29)], (501.25, 300.0),
                (1e-38, -2e-38, 0.0, 1e-35, -5e-36, 2000.0), 1e-16, 1e-16),
    # stages far beyond 2^60: a start within rounding of a well
    "stage_overflow": ([(500.0, 300.0, 0.25, 1e30), (900.0, 650.0, 0.25, 400.0)],
                       (500.0 + 2.0 ** -40, 300.0), COEF, 0.25, 20.0),
}


@pytest.mark.parametrize("case", sorted(RULES))
def test_short_division_rules_bit_exact_vs_oracle(gpu_ctx, case):
    wells, start, coef, por, thick = RULES[case]
    w = np.array(wells, dtype=float)
    xo, yo = w[0, 0], w[0, 1]
    real = Realizations([10.0], [por], [thick], w[:, 3].reshape(1, -1), np.array(coef, float))
    om = O.OracleModel(0.0, 10.0, por, thick, w, xo, yo, coef)
    cap = 400
    verts, nverts, status = trace_vertices(np.ascontiguousarray(w[:, :2]), xo, yo, real,
                                           np.array([start]), 300.0, 1.0, 10.0, True, cap)
    ov, res = om.backtrace(start[0], start[1], 300.0, 1.0, 10.0, confined=True, max_steps=cap)
    assert (status[0], nverts[0]) == (res.status, res.nverts)
    assert np.array_equal(verts[0, :nverts[0]], ov)
    assert np.array_equal(np.signbit(verts[0, :nverts[0]]), np.signbit(ov))


@pytest.mark.parametrize("tol,maxstep", [(1e-9, 10.0), (1e-4, 3.0), (0.02, 1e4), (1e-300, 1.0),
                                         (1.0, 1e-3)])
def test_step_factor_rules_bit_exact_vs_oracle(gpu_ctx, tol, maxstep):
    """The step factor by the power (a tight tolerance), by the step length
    (a short maxstep) and on either side of the rule between them."""
    w = np.array([(0.0, 0.0, 0.25, 700.0), (150.0, 80.0, 0.25, 400.0), (-90.0, 60.0, 0.25, -300.0)])
    real = Realizations([10.0], [0.25], [20.0], w[:, 3].reshape(1, -1), np.array(COEF, float))
    om = O.OracleModel(0.0, 10.0, 0.25, 20.0, w, 0.0, 0.0, COEF)
    cap = 1500
    for start in ((1.25, 0.5), (149.0, 80.5), (-90.0, 61.0)):
        verts, nverts, status = trace_vertices(np.ascontiguousarray(w[:, :2]), 0.0, 0.0, real,
                                               np.array([start]), 2000.0, tol, maxstep, True, cap)
        ov, res = om.backtrace(start[0], start[1], 2000.0, tol, maxstep, confined=True,
                               max_steps=cap)
        assert (status[0], nverts[0]) == (res.status, res.nverts)
        assert np.array_equal(verts[0, :nverts[0]], ov)


def _worst_numerators(k):
    """Mantissas (of 53 bits) whose quotients by b = 2 - k 2^-52 lie closest to
    the middle of two doubles: 2^54 A = r (mod 2^53 - k) for small odd r."""
    b = 2 ** 53 - k
    inv = pow(2 ** 54, -1, b)
    out = [r * inv % b for r in (1, -1, 3, -3, 5, -5, 7, -7)]
    return [a for a in out if a > b // 2]


def test_quotients_by_divisors_just_below_a_power_of_two(gpu_ctx):
    """thickness x porosity = 2 - k 2^-52 for odd k, where a reciprocal that is
    not the nearest double gives the wrong quotient for the numerators used
    here, the regional discharges: the vertices are the oracle's, whose
    division is IEEE's."""
    cases = [(k, a) for k in (1, 3, 5, 7, 9, 11, 13, 25, 33, 35, 999, 4001, 65535, 65537)
             for a in _worst_numerators(k)]
    # numerators a * 2^-52 and, along y, the next case's
    d = np.array([a * 2.0 ** -52 for _, a in cases])
    thick = np.array([(2 ** 53 - k) * 2.0 ** -51 for k, _ in cases])
    e = np.array([cases[(i + 1) % len(cases)][1] * -2.0 ** -53
                  if cases[(i + 1) % len(cases)][0] == k else 0.0
                  for i, (k, _) in enumerate(cases)])
    n = len(cases)
    w = np.array([(500.0, 300.0, 0.25, 0.0)])
    coef = np.zeros((n, 6))
    coef[:, 3], coef[:, 4] = d, e
    real = Realizations(np.full(n, 10.0), np.full(n, 0.5), thick, np.zeros((n, 1)), coef)
    verts, nverts, status = trace_vertices(np.ascontiguousarray(w[:, :2]), 0.0, 0.0, real,
                                           np.zeros((1, 2)), 50.0, 1.0, 10.0, True, 40)
    for i, (k, _) in enumerate(cases):
        om = O.OracleModel(0.0, 10.0, 0.5, thick[i], w, 0.0, 0.0, tuple(coef[i]))
        ov, res = om.backtrace(0.0, 0.0, 50.0, 1.0, 10.0, confined=True, max_steps=40)
        assert (status[i], nverts[i]) == (res.status, res.nverts), k
        assert np.array_equal(verts[i, :nverts[i]], ov), k
