"""The slot table of the wave-per-source search on the CPU (tests/slot_table_check.cpp over
relearn_amd/csrc/rl_slot_table.h): traversals that need up to 2,047 slots end with the records and masses of
their tree, larger ones are handed over, and the pull of the masses always makes progress."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MOST = 2047


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("slots") / "slot_table_check")
    cxx = os.environ.get("CXX", shutil.which("g++") or "g++")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Wextra", "-I", os.path.join(ROOT, "relearn_amd", "csrc"),
                    os.path.join(ROOT, "tests", "slot_table_check.cpp"), "-o", exe], check=True)

    def run(slots, waiting, seed, end_full=False):
        cmd = [exe, str(slots), str(waiting), str(seed)] + (["--end-full"] if end_full else [])
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=20)
        assert r.returncode == 0, (cmd, r.stdout)
        return r.stdout.split()

    return run


# the table's end, and the ring emptied at each multiple of 64
@pytest.mark.parametrize("slots", [1, 2, 64, 511, 512, 513, 575, 576, 577, 1024, 1983, 1984, 1985, 2045, 2046, 2047,
                                   2048, 2049, 2111, 2112, 2113])
@pytest.mark.parametrize("waiting", [1, 8, 64, 400])
def test_slot_table_ends(check, slots, waiting):
    for seed in range(8):
        for end_full in (False, True):
            assert check(slots, waiting, seed, end_full)[0] == ("done" if slots <= MOST else "overflow")


# more waiting slots than the ring holds: they wait in the table
@pytest.mark.parametrize("slots", [600, 1024, 2046, 2047, 2048, 2049])
@pytest.mark.parametrize("waiting", [447, 448, 449, 504, 512, 520, 600, 1000, 2000])
def test_slots_that_wait_outside_the_ring(check, slots, waiting):
    for seed in range(8):
        kind, _, most = check(slots, waiting, seed)
        assert kind == ("done" if slots <= MOST else "overflow")
        if slots >= MOST - 1:
            assert int(most) >= min(waiting, 1200)
