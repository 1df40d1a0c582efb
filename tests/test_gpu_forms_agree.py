"""The two part shapes of the FP64 stage kernel (16x4x2, form 1, and 16x4x4, form 2) evaluate the same
arithmetic per cell: right-hand sides and whole steps agree bit for bit, in vacuum and with matter. So
do the mixed form's steps with every tile in FP64 (its own launch of the large parts, last stage
included) and the FP64 form's, at extents off the parts' edges; and with the default threshold a
block away from the puncture really is stepped in FP32."""
import numpy as np
import pytest

from golden_cases import sources
from oracle.oracle import Geom, group_rel

pytestmark = pytest.mark.gpu


def bits(a):
    return np.ascontiguousarray(a).view(np.uint64)


@pytest.mark.parametrize("matter", [False, True])
@pytest.mark.parametrize("n", [(16, 4, 8), (18, 9, 7), (40, 20, 23), (64, 48, 40)])
def test_part_shapes_agree(engine, oracle, n, matter):
    import granite_amd as ga
    from hipmem import DeviceArray

    h = 0.125
    lo = [-0.5 * h * v + 0.01 for v in n]
    g = Geom(n, 4, lo, [a + h * v for a, v in zip(lo, n)])
    u = oracle.add_noise(g, oracle.init_bl(g, [1.0], [[0.05, -0.02, 0.01]]), 23, 1e-3, range(22))
    dev = [DeviceArray(a) for a in sources(g, 5)] if matter else []
    p, outs = ga.CCZ4Params(), []
    for form in (1, 2, 1):
        blk = ga.GridBlock(0, 0, g.n, g.lo, g.hi, g.ng)
        blk.array[...] = u
        lvl = ga.Level([blk], engine)
        lvl.upload()
        if matter:
            lvl.set_sources(0, *[d.data_ptr() for d in dev])
        lvl.set_tuning(ga.TUNE_STAGE, 0, form)
        print(f"[gpu] form {form} {n} matter {matter}", flush=True)
        rhs = lvl.rhs(0, p)
        for step in range(3):
            lvl.rk3_step(p, 0.02, pre_fill=ga.BC_OUTFLOW, use_graph=step > 0)
        lvl.download()
        outs.append((bits(rhs), bits(blk.array)))
        assert np.isfinite(blk.array).all()
        lvl.close()
    for other in outs[1:]:
        for a, b in zip(outs[0], other):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [(5, 7, 3), (17, 5, 9), (33, 20, 12), (48, 9, 25)])
def test_mixed_steps_at_the_edges_of_parts(engine, oracle, n):
    import granite_amd as ga

    h = 0.25
    geoms = []
    for off in (6.0, 0.0):  # away from the puncture, and on it
        lo = tuple(-h * v / 2 + off for v in n)
        geoms.append(Geom(n, 4, lo, tuple(a + h * v for a, v in zip(lo, n))))
    p, states = ga.CCZ4Params(), {}
    for name, precision, below in (("fp64", ga.PREC_FP64, 0.2), ("all fp64 tiles", ga.PREC_MIXED, 1e9),
                                   ("mixed", ga.PREC_MIXED, 0.2)):
        blks = []
        for i, g in enumerate(geoms):
            blk = ga.GridBlock(i, 0, g.n, g.lo, g.hi, g.ng)
            blk.array[...] = oracle.add_noise(g, oracle.init_bl(g, [1.0], [[0.0, 0.0, 0.0]]), 7 + i, 1e-4, range(22))
            blks.append(blk)
        lvl = ga.Level(blks, engine)
        lvl.upload()
        lvl.set_mixed_policy(below)
        print(f"[gpu] mixed steps {n}: {name}", flush=True)
        for step in range(2):
            lvl.rk3_step(p, 0.05, precision=precision, pre_fill=ga.BC_OUTFLOW, use_graph=step > 0)
        lvl.download()
        states[name] = [b.array.copy() for b in blks]
        lvl.close()
    for a, b, m in zip(states["fp64"], states["all fp64 tiles"], states["mixed"]):
        assert np.isfinite(a).all()
        assert np.array_equal(bits(a), bits(b))
        assert group_rel(m, a).max() < 1e-4
    assert not np.array_equal(states["mixed"][0], states["fp64"][0])
