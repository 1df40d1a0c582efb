"""The mixed form's parts at their edges: blocks smaller than a part, one cell over, odd rows, several
blocks in one launch. Bounds as for the mixed form's right-hand side (1e-4 of each tensor group);
with every tile in FP64 the result is the FP64 form's, bit for bit, whatever the split into parts."""
import numpy as np
import pytest

from oracle.oracle import Geom, group_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(5, 7, 3), (16, 4, 4), (17, 5, 9), (33, 20, 12), (48, 9, 25)])
def test_mixed_parts(engine, oracle, n):
    import granite_amd as ga

    h = 0.25
    blks, refs = [], []
    for i in range(2):  # away from the puncture (FP32 tiles) and on it
        lo = tuple(-h * v / 2 + (6.0 if i == 0 else 0.0) for v in n)
        g = Geom(n, 4, lo, tuple(a + h * v for a, v in zip(lo, n)))
        u = oracle.init_bl(g, [1.0], [[0.0, 0.0, 0.0]])
        oracle.rk3_step(g, u, 0.0625, 0)
        b = ga.GridBlock(i, 0, g.n, g.lo, g.hi, g.ng)
        b.array[...] = u
        blks.append(b)
        refs.append(oracle.rhs(g, u)[g.interior()])
    lvl = ga.Level(blks, engine)
    lvl.upload()
    p, I = ga.CCZ4Params(), g.interior()
    print(f"[gpu] mixed parts {n}", flush=True)
    for i in range(2):
        assert group_rel(lvl.rhs(i, p, ga.PREC_MIXED)[I], refs[i]).max() < 1e-4
    lvl.set_mixed_policy(1e9)
    for i in range(2):
        assert np.array_equal(lvl.rhs(i, p, ga.PREC_MIXED), lvl.rhs(i, p, ga.PREC_FP64))
    lvl.close()
