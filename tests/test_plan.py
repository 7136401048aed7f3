"""The rules that choose how many steps a launch or a barrier takes (lbm_plan.h)
against measured times: what they choose is not slower than one step at a time and
close to the best that was measured.  Times in microseconds a step, MI355X."""
import os
import subprocess

import pytest

from thesis_amd import lattices as LT

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "plan")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(HERE, "..", "thesis_amd", "csrc"),
                    os.path.join(HERE, "plan_main.cpp"), "-o", exe], check=True)

    def ask(line):
        r = subprocess.run([exe], input=line + "\n", capture_output=True, text=True, timeout=20)
        assert r.returncode == 0, line
        return [int(v) for v in r.stdout.split()]

    return ask


def time_of(times, steps, t):
    """The measured time at t steps; between two measured counts the longer one."""
    lo, hi = max(k for k in steps if k <= t), min(k for k in steps if k >= t)
    return max(times[steps.index(lo)], times[steps.index(hi)])


ONE, EIGHT, LARGE, MIX = "1 x 256x64", "8 x 256x64", "1 x 1024x256", "24 of a sweep"
HALOS = (1, 2, 3, 4, 5, 6, 8, 10)
# instances, steps between checks: at 1, 2, 3, 4, 5, 6, 8 and 10 steps a barrier
BATCH = {
    (ONE, 1): (12.1, 13.5, 14.2, 14.4, 14.2, 17.6, 18.8, 29.6),
    (ONE, 2): (9.8, 10.7, 11.2, 11.2, 11.2, 14.3, 14.5, 22.4),
    (ONE, 4): (8.5, 8.2, 6.4, 6.6, 7.1, 8.1, 8.5, 13.0),
    (ONE, 8): (8.0, 6.7, 5.6, 5.0, 5.2, 5.3, 4.7, 7.3),
    (ONE, 21): (7.5, 5.6, 4.4, 3.8, 3.6, 3.6, 3.5, 4.2),
    (ONE, 100): (7.3, 5.1, 3.8, 3.2, 3.1, 2.8, 2.6, 3.1),
    (EIGHT, 1): (34.6, 54.0, 54.1, 57.4, 55.5, 55.7, 57.3, 55.5),
    (EIGHT, 2): (27.6, 43.2, 41.7, 43.9, 42.8, 42.9, 44.5, 43.1),
    (EIGHT, 4): (23.3, 33.1, 24.6, 26.0, 26.6, 25.3, 27.4, 29.6),
    (EIGHT, 8): (21.6, 27.2, 21.4, 17.6, 19.5, 17.6, 14.1, 16.3),
    (EIGHT, 21): (20.3, 22.6, 16.7, 12.8, 12.4, 11.8, 10.4, 10.5),
    (EIGHT, 100): (19.8, 19.9, 14.2, 11.3, 9.6, 8.7, 8.0, 8.5),
    (LARGE, 1): (71.3, 69.5, 72.4, 71.1, 68.6, 73.4, 71.4, 68.1),
    (LARGE, 2): (56.2, 54.5, 54.0, 56.0, 54.7, 57.0, 56.6, 54.3),
    (LARGE, 4): (49.7, 39.6, 29.2, 30.4, 29.7, 30.3, 32.3, 35.1),
    (LARGE, 8): (43.2, 32.3, 25.9, 21.9, 22.3, 21.0, 18.6, 21.7),
    (LARGE, 21): (41.0, 26.4, 19.5, 15.0, 14.2, 14.2, 13.6, 14.6),
    (LARGE, 100): (40.4, 24.9, 17.3, 12.9, 11.9, 10.7, 10.5, 12.1),
    (MIX, 1): (111.7, 111.3, 115.2, 111.8, 111.5, 115.4, 111.8, 111.5),
    (MIX, 2): (90.5, 90.1, 92.8, 91.3, 90.5, 92.6, 90.3, 90.4),
    (MIX, 4): (80.0, 67.7, 54.4, 55.6, 57.9, 61.0, 71.3, 91.9),
    (MIX, 8): (74.8, 56.5, 47.7, 42.3, 45.0, 43.3, 45.8, 63.1),
    (MIX, 21): (71.7, 48.3, 38.4, 33.1, 32.5, 34.6, 40.0, 50.9),
    (MIX, 100): (69.8, 45.9, 34.3, 29.8, 29.6, 28.9, 35.0, 49.1),
}


@pytest.fixture(scope="module")
def shapes():
    return {ONE: [(256, 64)], EIGHT: [(256, 64)] * 8, LARGE: [(1024, 256)],
            MIX: [d["node_class"].shape[::-1] for d in LT.channel_sweep(24)]}


@pytest.mark.parametrize("name,every", BATCH)
def test_batch(plan, shapes, name, every):
    s = shapes[name]
    halo, squares, grid = plan(f"batch {len(s)} {every} " + " ".join(f"{x} {y}" for x, y in s))
    t = BATCH[name, every]
    assert 1 <= halo <= max(1, every - 1)
    side = 32 - 2 * halo
    assert squares == (0 if halo == 1 else sum(-(-x // side) * -(-y // side) for x, y in s))
    tiles = sum(-(-x * y // 1024) for x, y in s)
    assert grid == min(max(tiles, squares), 248)   # no workgroups, and so no barrier cost, without work
    assert time_of(t, HALOS, halo) <= 1.02 * t[0]
    assert time_of(t, HALOS, halo) <= 1.25 * min(t)
