"""The planner of the syncs on the CPU: its launches give the values, and write the
set of values, of the ops applied one after the other, also where solid surfaces
meet; a list of ops that it cannot follow to the end is refused, not shortened."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("sync_plan") / "sync_plan_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-ffp-contract=off", "-D_GLIBCXX_ASSERTIONS",
                    "-I", os.path.join(ROOT, "mpcns_mercury_amd", "csrc"), os.path.join(ROOT, "tests", "cpp", "sync_plan_check.cpp"),
                    "-o", exe], check=True)
    return lambda *a: subprocess.run([exe, *map(str, a)], capture_output=True, text=True, timeout=60)


# the launches: one more for each wall that reads what an earlier one sets
@pytest.mark.parametrize("g", [2, 4])
@pytest.mark.parametrize("blocks,launches", [
    ("6x5x4:", 1), ("6x5x4:0", 1), ("6x5x4:5", 1),
    ("6x5x4:01", 1),            # opposite walls, far enough from each other
    ("2x5x4:01", 2),            # two cells apart: each reads the other's first layer
    ("3x5x4:01", 1),            # three: both read the middle one, which neither sets
    ("6x5x4:02", 2), ("6x5x4:13", 2), ("6x5x4:35", 2),
    ("6x5x4:024", 3), ("2x2x2:012345", 6),
    ("6x5x4:0,5x5x5:2", 1),     # walls that do not meet: blocks of their own
    ("6x5x4:02,3x4x5:0,4x4x2:45", 3),  # blocks behind one whose walls meet
])
def test_launches_equal_the_ops_in_order(check, g, blocks, launches):
    r = check(g, blocks)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith(f"launches {launches} "), r.stdout


@pytest.mark.parametrize("blocks", ["6x5x4:02", "2x5x4:01", "6x5x4:02,6x5x4:0"])
def test_an_op_that_reads_what_it_sets_is_refused(check, blocks):
    r = check(2, blocks, "one_op")
    assert r.returncode == 3 and r.stdout.startswith("refused: "), r.stdout
