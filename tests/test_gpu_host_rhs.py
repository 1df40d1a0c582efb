"""The right-hand side on host arrays, on both of its routes (through pinned staging with one thread
or several, and directly where the block is larger than the staging): the interior equals the
level's right-hand side bit for bit, ghost cells of the result keep their values."""
import sys

import numpy as np
import pytest

from oracle.oracle import Geom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(5, 7, 3), (24, 25, 26), (40, 33, 37), (64, 48, 50), (96, 84, 80)])
@pytest.mark.parametrize("matter", [False, True])
def test_host_rhs_routes(engine, oracle, n, matter):
    import granite_amd as ga

    g = Geom(n, 4, (-1.0, -1.1, -0.9), (1.0, 0.9, 1.2))
    u = oracle.add_noise(g, oracle.init_bl(g, [1.0], [[0.1, 0.2, 0.3]]), 5, 1e-3, range(22))
    print(f"[gpu] host rhs {n} matter={matter}", flush=True)
    sys.stdout.flush()
    blk, out = ga.GridBlock(0, 0, g.n, g.lo, g.hi, g.ng), ga.GridBlock(1, 0, g.n, g.lo, g.hi, g.ng)
    blk.array[...] = u
    ev = ga.CCZ4Evolution(ga.CCZ4Params(), engine)
    N = g.stride
    # zero sources take the sources' kernel and give the vacuum result
    src = (np.zeros(N), np.zeros((N, 3)), np.zeros((N, 6)), np.zeros(N))
    lvl = ga.Level([blk], engine)
    lvl.upload()
    want = lvl.rhs(0, ga.CCZ4Params(), ga.PREC_FP64)
    I = g.interior()
    for rep in range(2):
        out.array[...] = 7.25 + rep
        if matter:
            ev.computeRHS(blk, out, *src)
        else:
            ev.computeRHSVacuum(blk, out)
        assert np.array_equal(out.array[I], want[I])
        mask = np.ones(out.array.shape[1:], bool)
        mask[I[1:]] = False
        assert np.all(out.array[:, mask] == 7.25 + rep)
        assert np.array_equal(blk.array, u)
    lvl.close()
