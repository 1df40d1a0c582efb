"""The native engine outlives what was made from it, whatever the order in which Python lets go of the
objects: every destroy call of a level, hierarchy or checkpoint comes before the engine's. Host-only,
on a stand-in for the library."""
import gc

import pytest

import granite_amd as ga
from granite_amd import ccz4


class Recorder:
    """Answers every entry point with success, hands out handles, keeps the destroy calls."""

    def __init__(self):
        self.destroyed = []
        self.made = 0

    def __getattr__(self, name):
        def call(*args):
            if name.endswith("_create"):
                self.made += 1
                args[-1]._obj.value = self.made
            if name.endswith("_destroy"):
                self.destroyed.append(name)
            return 0

        return call


@pytest.fixture
def lib(monkeypatch):
    r = Recorder()
    monkeypatch.setattr(ccz4, "library", lambda: r)
    return r


def parts():
    eng = ga.Engine(0)
    lvl = ga.Level([ga.GridBlock(0, 0, (4, 4, 4), (0.0,) * 3, (1.0,) * 3, 4)], eng)
    return eng, lvl, ga.Hierarchy([lvl], eng), ga.Checkpoint([lvl], eng)


@pytest.mark.parametrize("order", [(0, 1, 2, 3), (3, 0, 2, 1), (2, 3, 1, 0)])
def test_engine_goes_last_in_any_order_of_close(lib, order):
    objects = parts()
    for i in order:
        objects[i].close()
    assert sorted(lib.destroyed) == sorted(f"gr_{k}_destroy" for k in ("engine", "level", "hierarchy", "checkpoint"))
    assert lib.destroyed[-1] == "gr_engine_destroy"
    for o in objects:
        o.close()
    assert len(lib.destroyed) == 4


def test_engine_goes_last_from_a_cycle(lib):
    gc.disable()
    try:
        for _ in range(20):
            objects = list(parts())
            objects.append(objects)
    finally:
        gc.enable()
    del objects
    gc.collect()
    assert len(lib.destroyed) == 80
    live = 20 * 3
    alive = {"gr_level_destroy": 20, "gr_hierarchy_destroy": 20, "gr_checkpoint_destroy": 20}
    engines = 0
    for name in lib.destroyed:
        if name == "gr_engine_destroy":
            engines += 1
        else:
            alive[name] -= 1
            live -= 1
        # an engine that is gone has taken its three parts before it
        assert engines * 3 <= 60 - live
    assert engines == 20 and not any(alive.values())
