"""Small structure on a background value in the fields whose flat value is zero (K, Theta, Gamma-hat,
A~, the shift): the cell's dissipation keeps the reference's order, bit for bit, and its advection
is as accurate as plain double arithmetic."""
import numpy as np
import pytest

from oracle.oracle import Geom
from test_host_cell_math import hcell  # noqa: F401  (fixture)


@pytest.mark.parametrize("background", [0.2, 3.0])
def test_dissipation_order_of_every_field(oracle, hcell, background):  # noqa: F811
    # no lapse, no shift: the right-hand sides of these fields are the dissipation alone
    g = Geom((8, 7, 6), 4, (-1.0, -0.9, -0.8), (1.0, 0.9, 0.8))
    u = g.zeros()
    u[[0, 1, 4, 6]] = 1.0
    u[7:18] = background
    oracle.add_noise(g, u, 3, 1e-4, range(7, 18))
    I = g.interior()
    got, want = hcell(g, u)[I], oracle.rhs(g, u)[I]
    for v in range(7, 18):
        assert np.abs(want[v]).max() > 0.0
        assert np.array_equal(got[v], want[v]), v


@pytest.mark.parametrize("background", [0.2, 0.5, 3.0])
def test_shift_as_accurate_as_plain_double(hcell, oracle, background):  # noqa: F811
    # chi = 1 far above the blend's centre: w = 1 to rounding, the advection is the upwind sum. Both
    # errors are rounding of the same sums: taken over three fields of 960 cells their ratio is 1
    # to a few percent; 1.5 leaves room for a reordering of one sum, not for rounded weights.
    g = Geom((12, 10, 8), 4, (-1.5, -1.25, -1.0), (1.5, 1.25, 1.0))
    u = g.zeros()
    u[[0, 1, 4, 6, 18]] = 1.0
    u[19:22] = np.reshape([1.0, -0.7, 0.8], (3, 1, 1, 1)) * background
    oracle.add_noise(g, u, 5, 1e-6, range(19, 22))
    I = g.interior()
    b = u[19:22].astype(np.longdouble)
    h = (np.longdouble(hi) - np.longdouble(lo) for lo, hi in zip(g.lo, g.hi))
    w = np.longdouble(0.5) * (1 + np.tanh((np.longdouble(1.0) - np.longdouble(0.05)) / np.longdouble(0.02)))
    want = 0 * b
    for d, L in enumerate(h):
        dx = L / g.n[d]
        t = {k: np.roll(b, -k, axis=3 - d) for k in range(-4, 5)}
        fwd = (-25 * b + 48 * t[1] - 36 * t[2] + 16 * t[3] - 3 * t[4]) / (12 * dx)
        bwd = -(-25 * b + 48 * t[-1] - 36 * t[-2] + 16 * t[-3] - 3 * t[-4]) / (12 * dx)
        cen = (-t[2] + 8 * t[1] - 8 * t[-1] + t[-2]) / (12 * dx)
        be = b[d]
        want = want + be * (w * np.where(be >= 0, bwd, fwd) + (1 - w) * cen)
        ko = t[-3] + t[3] - 6 * (t[-2] + t[2]) + 15 * (t[-1] + t[1]) - 20 * b
        want = want + np.longdouble(0.1) / (64 * dx) * ko
    err = [np.sqrt(np.mean((f(g, u, eta=0.0)[I][19:22].astype(np.longdouble) - want[I]) ** 2)) for f in (hcell, oracle.rhs)]
    assert err[1] < 1e-12 * background
    assert err[0] <= 1.5 * err[1], [float(e) for e in err]
