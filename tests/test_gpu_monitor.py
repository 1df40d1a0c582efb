"""The constraint monitor at the edges of its parts, against the oracle: H and M_i per cell (ghosts
zero) and their sums over the interior. Extents one off a 16x4x4 part, odd rows, more ghosts than
the stencils reach, and a block with more parts (640) than the 512 workgroups of the sums."""
import numpy as np
import pytest

from oracle.oracle import Geom

pytestmark = pytest.mark.gpu

TOL = 1e-12  # the FP64 parity bar


@pytest.mark.parametrize("n,ng", [((1, 1, 1), 4), ((17, 5, 3), 4), ((15, 4, 9), 5), ((64, 64, 40), 4)])
def test_monitor_against_oracle(engine, oracle, n, ng):
    import granite_amd as ga

    h = 0.25
    lo = [-0.5 * h * v + 0.03 for v in n]
    g = Geom(n, ng, lo, [a + h * v for a, v in zip(lo, n)])
    u = oracle.add_noise(g, oracle.init_bl(g, [1.0], [[0.05, -0.02, 0.01]]), 29, 1e-2, range(22))
    blk = ga.GridBlock(0, 0, g.n, g.lo, g.hi, g.ng)
    blk.array[...] = u
    print(f"[gpu] monitor {n} ng {ng}", flush=True)
    ham, mom = ga.CCZ4Evolution(ga.CCZ4Params(), engine).computeConstraints(blk)
    rh, rm = oracle.constraints(g, u)
    assert np.max(np.abs(ham.reshape(rh.shape) - rh)) < TOL * np.max(np.abs(rh))
    assert np.max(np.abs(mom.reshape(rm.shape) - rm)) < TOL * np.max(np.abs(rm))
    lvl = ga.Level([blk, blk], engine)
    lvl.upload()
    s, cnt = lvl.constraints_l2()
    want = 2.0 * float(np.sum(rh * rh))
    assert cnt == 2 * int(np.prod(n)) and abs(s - want) < TOL * want
    lvl.close()
