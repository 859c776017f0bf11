"""The tiled kernel of the discounted return and its gradient (mrb_returns.h), run on the CPU with lanes that run one after the
other between the places where a wave or a workgroup meets (tests/host_wave/returns): what a lane takes from LDS that another
lane of its wave has put there has to lie behind such a place. Every form of the kernel, bit for bit against the recurrence."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests", "host_wave", "returns")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    at = tmp_path_factory.mktemp("returns")
    with open(os.path.join(ROOT, "mindrl_amd", "csrc", "mrb_returns.h")) as f:
        text = f.read()
    # (the register constraint of an empty statement that hides an address from the compiler is the device's)
    text, hidden = re.subn(r'asm volatile\(""[^;]*;', "", text.replace("#include <hip/hip_runtime.h>\n", ""))
    assert hidden == 1
    (at / "mrb_returns.h").write_text(text)
    for name in ("mrb_device.h", "returns.cpp"):
        with open(os.path.join(HERE, name)) as f:
            (at / name).write_text(f.read())
    out = at / "returns"
    res = subprocess.run(["/opt/rocm/llvm/bin/clang++", "-O1", "-U_FORTIFY_SOURCE", "-std=c++17", "-Wall", "-Wno-unknown-attributes", "-ffp-contract=off",
                          "-o", str(out), str(at / "returns.cpp")], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    return str(out)


@pytest.mark.parametrize("what", ["quads", "columns", "wide"])
def test_lanes_in_any_order(program, what):
    res = subprocess.run([program, what], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert res.returncode == 0, res.stdout
