"""Captured steps whose key changes from call to call, with no wait between the calls: every result is
that of the eager step, bit for bit. A graph is dropped only after its last launch has ended."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def levels(engine, n=3, shift=0.0):
    import granite_amd as ga

    out = []
    for i in range(n):
        dx = 0.25 / 2 ** i
        size = (16 + 8 * i, 8, 12)
        lo = (-0.5 * dx * size[0] + shift, -0.4, -0.5)
        blks = [ga.GridBlock(k, 0, size, tuple(a + 3.0 * k for a in lo),
                             tuple(a + 3.0 * k + dx * m for a, m in zip(lo, size)), 4) for k in range(2)]
        lvl = ga.Level(blks, engine)
        lvl.init_brill_lindquist([1.0], [[0.05, 0.02, 0.01]])
        out.append((lvl, blks, 0.25 * dx))
    return out


def same(a, b):
    for (la, ba, _), (lb, bb, _) in zip(a, b):
        la.download()
        lb.download()
        for x, y in zip(ba, bb):
            assert np.isfinite(x.array).all()
            assert np.array_equal(x.array, y.array)
        la.close()
        lb.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_alternating_level_sets(engine, precision):
    import granite_amd as ga

    p = ga.CCZ4Params()
    captured, eager = levels(engine), levels(engine)
    sets = ([0, 1, 2], [2, 0], [1], [0, 1, 2])
    print(f"[gpu] alternating level sets, precision {precision}", flush=True)
    for use_graph, lv in ((True, captured), (False, eager)):
        for which in sets * 2:
            ga.levels_rk3_step([lv[i][0] for i in which], [lv[i][2] for i in which], p, precision=precision,
                               pre_fill=ga.BC_OUTFLOW, use_graph=use_graph)
    same(captured, eager)


@pytest.mark.parametrize("precision", [0, 1])
def test_level_step_with_changing_dt(engine, precision):
    import granite_amd as ga

    p = ga.CCZ4Params()
    captured, eager = levels(engine, 1), levels(engine, 1)
    print(f"[gpu] changing dt, precision {precision}", flush=True)
    for use_graph, lv in ((True, captured), (False, eager)):
        for step in range(8):
            lv[0][0].rk3_step(p, lv[0][2] * (1.0 - 0.05 * step), precision=precision, pre_fill=ga.BC_OUTFLOW,
                              use_graph=use_graph)
    same(captured, eager)


def test_hierarchy_step_with_changing_dt(engine):
    import granite_amd as ga

    p = ga.CCZ4Params()
    results = []
    print("[gpu] hierarchy, changing dt", flush=True)
    for use_graph in (True, False):
        blks = [[ga.GridBlock(0, 0, (16, 16, 16), (-8.0,) * 3, (8.0,) * 3, 4)],
                [ga.GridBlock(0, 1, (16, 12, 8), (-4.0, -3.0, -2.0), (4.0, 3.0, 2.0), 4)]]
        lv = [ga.Level(b, engine) for b in blks]
        for level in lv:
            level.init_brill_lindquist([0.5, 0.5], [[-1.0, 0.0, 0.0], [1.0, 0.0, 0.0]])
        H = ga.Hierarchy(lv, engine)
        for step in range(4):
            H.step(p, 0.25 * (1.0 - 0.1 * step), use_graph=use_graph)
        for level in lv:
            level.download()
        results.append([b[0].array.copy() for b in blks])
        H.close()
        for level in lv:
            level.close()
    for a, b in zip(*results):
        assert np.isfinite(a).all() and np.array_equal(a, b)
