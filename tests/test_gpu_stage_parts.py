"""The FP64 stage kernel's part shapes at the edges of their tiles, against the oracle.

Parts are 16x4x2 or 16x4x4 cells, the halo staged by 16-byte loads: rows of odd length (whose
pairs are aligned to 8 bytes only), extents one off a part, single cells, more ghosts than the
stencils reach, and launches either side of the size where the large parts take over (64 launch
tiles of 16x4x8), in vacuum and with matter sources."""
import numpy as np
import pytest

from golden_cases import sources
from oracle.oracle import Geom, group_rel

pytestmark = pytest.mark.gpu

TOL = 1e-12  # the FP64 parity bar: agreement is round-off of one evaluation


@pytest.mark.parametrize("n,ng,matter", [
    ((1, 1, 1), 4, False),
    ((15, 5, 3), 4, False),
    ((17, 3, 9), 4, True),
    ((16, 4, 2), 5, False),
    ((31, 9, 5), 5, True),
    ((33, 8, 4), 4, False),
    ((63, 15, 31), 4, False),   # 64 tiles: the last small launch
    ((65, 17, 21), 4, True),    # 75 tiles: large parts, odd rows
    ((80, 13, 27), 6, False),   # large parts, wide ghosts
])
def test_parts_against_oracle(engine, oracle, n, ng, matter):
    import granite_amd as ga
    from hipmem import DeviceArray

    h = 0.25
    lo = [-0.5 * h * v + 0.03 for v in n]
    g = Geom(n, ng, lo, [a + h * v for a, v in zip(lo, n)])
    # noise large enough that no right-hand side of a one-cell block is a cancellation of O(1) terms
    u = oracle.add_noise(g, oracle.init_bl(g, [1.0], [[0.05, -0.02, 0.01]]), 23, 1e-2, range(22))
    blk = ga.GridBlock(0, 0, g.n, g.lo, g.hi, g.ng)
    blk.array[...] = u
    lvl = ga.Level([blk], engine)
    lvl.upload()
    host = dev = None
    if matter:
        host = sources(g, 5)
        dev = [DeviceArray(a) for a in host]
        lvl.set_sources(0, *[d.data_ptr() for d in dev])
    p = ga.CCZ4Params()
    print(f"[gpu] parts {n} ng {ng} matter {matter}", flush=True)
    I = g.interior()
    assert group_rel(lvl.rhs(0, p)[I], oracle.rhs(g, u, sources=host)[I]).max() < TOL
    lvl.rk3_step(p, 0.0625, pre_fill=ga.BC_OUTFLOW)
    lvl.download()
    ref = oracle.fill_ghosts(g, u.copy(), 2)
    oracle.rk3_step(g, ref, 0.0625, 0, sources=host)
    assert group_rel(blk.array, ref).max() < TOL
    lvl.close()
