"""Which batches are stored through the L2 (mrb_rows.h): the rule is the host's, so it is looked at here. Gathers from beyond the size that the
dies' caches hold, samples from 20 MB on."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MB = 1 << 20


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = tmp_path_factory.mktemp("rules") / "through"
    res = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                          "-I", os.path.join(ROOT, "mindrl_amd", "csrc"), "-o", str(out), os.path.join(ROOT, "tests", "host_rules", "through.hip")],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    return str(out)


def through(program, size):
    """(a sample, a gather)"""
    res = subprocess.run([program, str(size)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert res.returncode == 0
    return tuple(int(c) for c in res.stdout.strip())


def test_what_the_caches_hold_stays_there_for_its_reader(program):
    assert through(program, 20 * MB) == (0, 0)
    assert through(program, 20 * MB + 1) == (1, 0)
    assert through(program, 40 * MB) == (1, 0)
    assert through(program, 40 * MB + 1) == (1, 1)
