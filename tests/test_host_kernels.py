"""The kernels of the source files that tests/test_host_cpu.py does not look at: no scratch memory, no more registers than
their workgroups' waves have, the LDS their comments state."""
import os
import re
import subprocess

import pytest


@pytest.mark.parametrize("source,count", [("mrb_range_one.hip", 10), ("mrb_short.hip", 5), ("mrb_push_many.hip", 3), ("mrb_samples_large.hip", 4), ("mrb_silent.hip", 1)])
def test_kernels_use_no_scratch_memory(source, count, tmp_path):
    from mindrl_amd import build
    out = tmp_path / "kernels.s"
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    res = subprocess.run(["/opt/rocm/bin/hipcc"] + flags + ["--cuda-device-only", "-S", "-o", str(out), os.path.join(build.CSRC, source)],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    kernels = {}
    for block in out.read_text().split("  - .agpr_count:")[1:]:
        number = lambda key: int(re.search(r"\.%s:\s+(\d+)" % key, block).group(1))
        kernels[re.search(r"\.name:\s+(\S+)", block).group(1)] = (
            number("private_segment_fixed_size"), number("group_segment_fixed_size"), number("vgpr_count"))
    assert len(kernels) == count, sorted(kernels)
    for name, (scratch, lds, vgprs) in kernels.items():
        assert scratch == 0 and vgprs <= 128, (name, scratch, vgprs)
        runs = re.search(r"k_range_one(?:_push)?ILi(\d+)", name)
        if not runs:  # a tile's leaves, or three levels of a pair of roots and a mark per wave
            assert lds <= 1088, (name, lds)
            continue
        # the election words, a root of each tree and a mark per tile, a mark per run and a word per wave
        leaves = 1 << int(runs.group(1))
        assert 0 <= lds - (8 * leaves + 12 * (leaves // 256)) <= 1088, (name, lds)


@pytest.mark.parametrize("source", ["mrb.hip", "mrb_short.hip", "mrb_returns.hip", "mrb_samples_large.hip"])
def test_stores_written_in_assembly_keep_their_registers(source, tmp_path):
    """A 16-byte store's registers may be written two wait states behind it, which the compiler does not look after in inline assembly."""
    from mindrl_amd import build
    out = tmp_path / "kernels.s"
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    res = subprocess.run(["/opt/rocm/bin/hipcc"] + flags + ["--cuda-device-only", "-S", "-o", str(out), os.path.join(build.CSRC, source)],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    written = re.findall(r";;#ASMSTART\n(.*?);;#ASMEND", out.read_text(), re.S)
    stores = [text for text in written if "store_dwordx4" in text]
    assert stores
    for text in stores:
        assert re.search(r"store_dwordx4 [^\n]*\n\s*s_nop ([1-9])", text), text
