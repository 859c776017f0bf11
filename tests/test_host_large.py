"""Which fields a sample of many rows copies by themselves (mrb_lds_sample.h): the rule is the host's, so it is looked at here. Not those
of buffers whose rows come from the caches, where that copy was slower than the one by a look-up for each granule."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MB = 1 << 20


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = tmp_path_factory.mktemp("rules") / "large"
    res = subprocess.run(["/opt/rocm/bin/hipcc", "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                          "-I", os.path.join(ROOT, "mindrl_amd", "csrc"), "-o", str(out), os.path.join(ROOT, "tests", "host_rules", "large.hip")],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    return str(out)


@pytest.mark.parametrize("row,strata,nbatch,size,line", [
    (2048, 16, 1, 25 * MB, 0), (2048, 16, 1, 64 * MB, 0), (2048, 16, 1, 64 * MB + 1, 56 * MB), (4096, 32, 1, 2000 * MB, 56 * MB),
    (2048, 16, 2, 64 * MB, 24 * MB), (1024, 64, 5, 64 * MB, 24 * MB), (1024, 64, 5, 64 * MB + 1, 56 * MB),
    (2049, 16, 1, 25 * MB, 144 * MB), (2040, 16, 5, 64 * MB, 144 * MB), (1101, 64, 1, 96 * MB, 144 * MB), (131, 256, 1, 64 * MB, 144 * MB)])
def test_by_what_the_rows_held_take(program, row, strata, nbatch, size, line):
    took = [subprocess.run([program, str(row), str(strata), str(nbatch), str(size), str(held)], stdout=subprocess.PIPE, text=True, timeout=60).stdout
            for held in (line, line + 1, 1 << 40)]
    assert took == ["0\n", "1\n", "1\n"]


@pytest.mark.parametrize("row,strata,size,large", [
    (128, 256, 16 * MB, 1), (127, 256, 16 * MB, 1), (112, 256, 16 * MB, 0), (512, 64, 64 * MB, 1), (496, 64, 64 * MB, 0),
    (2048, 16, 25 * MB, 1), (2032, 16, 25 * MB, 0), (1024, 16, 25 * MB, 0), (2049, 16, 96 * MB + 1, 0), (1, 256, 16 * MB, 0)])
def test_by_a_workgroups_granules(program, row, strata, size, large):
    assert subprocess.run([program, str(row), str(strata), "1", str(size), str(5 * MB if row % 16 == 0 else 1 << 40)], stdout=subprocess.PIPE, text=True,
                          timeout=60).stdout == "%d\n" % large
