"""The tuner times each of the stage kernel's part shapes once: the form that a launch of this size takes
by itself stands for the fixed form of the same shape, so noise does not choose between them."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,alias", [((16, 8, 8), 1), ((32, 32, 32), 1), ((64, 48, 40), 2)])
def test_forms_of_one_kernel_share_a_time(engine, n, alias):
    import granite_amd as ga

    ga.tune_clear()
    lvl = ga.Level([ga.GridBlock(0, 0, n, (0.0,) * 3, tuple(0.25 * v for v in n), 4)], engine)
    lvl.init_brill_lindquist([1.0], [[0.1, 0.2, 0.3]])
    print(f"[gpu] tune {n}", flush=True)
    t = lvl.autotune(ga.CCZ4Params(), 0.05)["stage"][0]
    assert t[alias] == t[0] and t[3 - alias] > 0
    assert lvl.tuning(ga.TUNE_STAGE, 0) == (0 if t[0] <= t[3 - alias] else 3 - alias)
    lvl.close()
    ga.tune_clear()
