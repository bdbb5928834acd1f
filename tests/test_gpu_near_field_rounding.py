"""The regularized near field rounds rho^2 = r^2 / sij^2 as a division does.

One source at the origin, targets on the axes, distances and sizes of few bits
(so that their squares are exact), one box: every other operation of the algebraic
kernel's pair is a single rounding, so numpy repeats the velocity bit for bit.
(With r^2 times a rounded reciprocal of sij^2 a quarter of the quotients are off
in the last place.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_pair_quotient_is_the_division(gpu):
    from lsmps_vpm_v2_amd import FmmSolver
    g = np.random.default_rng(5)
    n = 4000
    r = g.integers(1, 65, n) / 64.0
    on_x = g.random(n) < 0.5
    r[:2], on_x[:2] = 1.0, (True, False)  # a square field
    x, y = np.where(on_x, r, 0.0), np.where(on_x, 0.0, r)
    s = g.integers(3, 1000, n) / 64.0
    x, y, s = np.append(x, 0.0), np.append(y, 0.0), np.append(s, 0.75)
    gz = np.append(np.zeros(n), 0.37)
    u, v = FmmSolver(u_inf=0.0, v_inf=0.0).velocity_type1(x, y, s, gz, n_s=4096, lmax=2, ndp=4,
                                                          icutoff=1)
    rho2 = (r * r) / (0.25 * (s[:n] ** 2 + s[n] ** 2))
    q = 0.37 * (-1.0 / (2.0 * np.pi))
    e = (q * (1.0 / (r * r))) * ((rho2 * (rho2 + 2.0)) / ((rho2 + 1.0) * (rho2 + 1.0))) * r
    np.testing.assert_array_equal(u[:n], np.where(on_x, 0.0, e))
    np.testing.assert_array_equal(v[:n], np.where(on_x, -e, 0.0))
