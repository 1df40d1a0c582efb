"""The 1/r ghost fill at the ends of the number range, bit for bit against the oracle: fall-offs whose
quotients come near the smallest normal number, or overflow, and infinities, beside ordinary values
and zeros. (No subnormal values: a library built with -ffast-math flushes them in its whole process, so
the oracle's depend on the tests that ran before.)"""
import numpy as np
import pytest

from oracle.oracle import Geom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", [1, 2])  # the launch of one block, and that of several
@pytest.mark.parametrize("groups", [1, 4, 11])
@pytest.mark.parametrize("scale", [2.0 ** -1016, 2.0 ** -960, 1.0, 2.0 ** 1019, 2.0 ** 1022, np.inf])
def test_sommerfeld_over_the_range(engine, oracle, blocks, groups, scale):
    import granite_amd as ga

    g = Geom((13, 9, 11), 4, (-0.7, -0.4, 0.2), (1.1, 0.6, 1.6))
    rng = np.random.default_rng(5)
    blks, states = [], []
    for i in range(blocks):
        u = rng.uniform(0.5, 2.0, g.zeros().shape) * rng.choice([-1.0, 1.0], g.zeros().shape)
        u[::3] = rng.choice([0.0, -0.0, 1.0], u[::3].shape)
        u[rng.random(u.shape) < 0.5] *= scale  # ordinary values beside the extreme ones
        blk = ga.GridBlock(i, 0, g.n, g.lo, g.hi, g.ng)
        blk.array[...] = u
        blks.append(blk)
        states.append(u)
    lvl = ga.Level(blks, engine)
    lvl.upload()
    lvl.set_tuning(ga.TUNE_GHOST, 0, groups)
    print(f"[gpu] ghost fill, {blocks} blocks, {groups} groups, scale {scale}", flush=True)
    lvl.fill_ghosts(ga.BC_SOMMERFELD)
    lvl.download()
    for blk, u in zip(blks, states):
        want = oracle.fill_ghosts(g, u.copy(), 0)
        assert np.array_equal(blk.array, want, equal_nan=True)
        ok = ~np.isnan(want)
        assert np.array_equal(np.signbit(blk.array[ok]), np.signbit(want[ok]))
    lvl.close()
