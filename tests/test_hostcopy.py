"""The staging of field copies on a CPU stand-in for the runtime (tests/hostcopy):
what one card cannot show, a context whose device is not the caller's current one,
and what must not be provoked there."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "thesis_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("hostcopy") / "check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", os.path.join(HERE, "hostcopy"), "-I", CSRC,
                    os.path.join(HERE, "hostcopy", "check.cpp"), os.path.join(CSRC, "lbm_hostcopy.cpp"), "-o", exe],
                   check=True)
    return lambda case: subprocess.run([exe, case], capture_output=True, text=True, timeout=60)


def holds(r):
    assert r.returncode == 0, r.stdout + r.stderr


def test_context_of_another_device(check):
    holds(check("device"))


def test_host_memory_runs_out(check):
    holds(check("memory"))


def test_pinned_memory_and_events_run_out(check):
    holds(check("errors"))


def test_pinned_destination(check):
    holds(check("pinned"))
