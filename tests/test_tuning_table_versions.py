"""A tuning table written by an earlier version of the library names stagings of the stage kernel that no
longer exist: its stage entries are checked but not taken, all others are. Host-only."""
import os

import pytest

import granite_amd as ga
from test_tuning_table import _lib

OLD = "# granite-ccz4 tuning table: kind class precision value\n"


def rows(path):
    ga.tune_save(path)
    return sorted(tuple(ln.split()) for ln in open(path) if not ln.startswith("#"))


def test_stage_entries_of_an_old_table_are_not_taken(tmp_path):
    _lib()
    ga.tune_clear()
    path, out = os.path.join(str(tmp_path), "old.txt"), os.path.join(str(tmp_path), "out.txt")
    with open(path, "w") as f:
        f.write(OLD + "0 0 0 1\n0 3 0 2\n1 2 0 11\n2 1 0 2\n")
    ga.tune_load(path)
    assert rows(out) == [("1", "2", "0", "11"), ("2", "1", "0", "2")]
    ga.tune_clear()


def test_a_current_table_is_taken_whole(tmp_path):
    _lib()
    ga.tune_clear()
    path, out = os.path.join(str(tmp_path), "new.txt"), os.path.join(str(tmp_path), "out.txt")
    with open(path, "w") as f:  # no header: entries by hand, in the current numbers
        f.write("0 0 0 1\n0 3 0 2\n1 2 0 11\n")
    ga.tune_load(path)
    want = rows(out)
    assert len(want) == 3
    ga.tune_clear()
    ga.tune_load(out)
    assert rows(path) == want
    ga.tune_clear()


def test_a_bad_stage_entry_still_rejects_an_old_table(tmp_path):
    _lib()
    path = os.path.join(str(tmp_path), "old.txt")
    with open(path, "w") as f:
        f.write(OLD + "0 0 0 3\n")
    with pytest.raises(ga.EngineError):
        ga.tune_load(path)
