"""An infinity in one cell reaches the same cells' right-hand sides as in the oracle: the weighted
sums of the merged advection and dissipation read no tap that the separate sums do not."""
import numpy as np
import pytest

from oracle.oracle import Geom
from test_host_cell_math import hcell  # noqa: F401  (fixture)


@pytest.mark.parametrize("sigma", [0.0, 0.1])
@pytest.mark.parametrize("field", [0, 1, 7, 13, 14, 17, 18, 19])
@pytest.mark.parametrize("shift", [0.3, -0.3, 0.0])
def test_infinity_reaches_the_same_cells(oracle, hcell, sigma, field, shift):  # noqa: F811
    g = Geom((9, 9, 9), 4, (-1, -1, -1), (1, 1, 1))
    u = oracle.add_noise(g, oracle.init_bl(g, [1.0], [[0.1, 0.2, 0.3]]), 3, 1e-3, range(22))
    u[19:22] = shift * (1 + u[19:22])
    u[field, 8, 8, 8] = np.inf
    I = g.interior()
    got, want = hcell(g, u, ko_sigma=sigma)[I], oracle.rhs(g, u, ko_sigma=sigma)[I]
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    assert not np.isfinite(want).all()
