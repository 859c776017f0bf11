"""How the workgroups of an update hand their roots to the last of them (mrb_meet.h), run on the CPU: waves of 64 lanes whose
operations on shared words come in any order and whose stores arrive late (tests/host_wave). Launches of 1 to 256 workgroups; counters
that hold anything, and a root that never comes, as two calls that change one buffer side by side can leave them; the launch
after the one with the last number."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = tmp_path_factory.mktemp("meet") / "meet"
    res = subprocess.run(["g++", "-O1", "-U_FORTIFY_SOURCE", "-std=c++17", "-Wall", "-Wno-unknown-pragmas", "-I", os.path.join(HERE, "host_wave"), "-o", str(out),
                          os.path.join(HERE, "host_wave", "meet.cpp")], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    return str(out)


@pytest.mark.parametrize("what", ["launches", "any_count", "missing_root", "last_number"])
def test_meeting(program, what):
    res = subprocess.run([program, what], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert res.returncode == 0, res.stdout
