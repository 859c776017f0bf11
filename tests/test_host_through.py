"""Which batches are stored through the L2 (mrb_rows.h): the rule is the host's, so it is looked at here. Gathers from beyond the size that the
dies' caches hold, samples from 20 MB on, and rows whose stores end within 64 bytes not beyond what the memory's cache takes."""
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


def through(program, size, rows, split=1, offset=0):
    """(by workgroups or waves: a sample, a gather; numbered over all rows: a gather, a sample)"""
    res = subprocess.run([program, str(size), str(split), str(offset)] + [str(r) for r in rows], stdout=subprocess.PIPE, text=True, timeout=60)
    assert res.returncode == 0
    return tuple(int(c) for c in res.stdout.strip())


@pytest.mark.parametrize("rows", [[28_224], [28_225], [2400, 600]])
def test_what_the_caches_hold_stays_there_for_its_reader(program, rows):
    assert through(program, 20 * MB, rows) == (0, 0, 0, 0)
    assert through(program, 20 * MB + 1, rows) == (1, 0, 0, 1)
    assert through(program, 40 * MB, rows) == (1, 0, 0, 1)
    assert through(program, 40 * MB + 1, rows) == (1, 1, 1, 1)
    assert through(program, 160 * MB, rows) == (1, 1, 1, 1)


@pytest.mark.parametrize("rows,split,offset,pieces,numbered", [
    ([28_224], 1, 0, 1, 1), ([4096, 64], 1, 0, 1, 1), ([40_960], 2, 0, 1, 1), ([40_192], 2, 0, 1, 1),   # whole pieces of 64 bytes
    ([28_192], 1, 0, 0, 1), ([2400], 1, 0, 0, 1), ([4096, 80], 1, 0, 0, 1),                             # a row ends within one
    ([40_000], 2, 0, 0, 1), ([33_600], 2, 0, 0, 1),                                                     # a workgroup's part does
    ([28_225], 1, 0, 0, 0), ([7500], 1, 0, 0, 0), ([4096, 17], 1, 0, 0, 0),                             # the granules themselves do
    ([28_224], 1, 16, 0, 0), ([28_224], 1, 4, 0, 0)])                                                   # the caller's matrix begins within one
def test_stores_that_end_within_64_bytes(program, rows, split, offset, pieces, numbered):
    for size in (160 * MB + 1, 1 << 32):
        assert through(program, size, rows, split, offset) == (pieces, pieces, numbered, numbered)
    assert through(program, 160 * MB, rows, split, offset) == (1, 1, 1, 1)
