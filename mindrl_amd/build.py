"""Builds libmrb.so (the HIP replay-buffer library) for gfx950 with hipcc, in-tree."""
import os
import subprocess
import sys

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
LIB = os.path.join(CSRC, "libmrb.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # every float/double operation rounds once, in source order (bit-exact tree and weights)
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    # no packed-fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-Wall",
]


SOURCES = ["mrb.hip", "mrb_returns.hip"]


def build(verbose=False):
    """Compile the sources of mindrl_amd/csrc into mindrl_amd/csrc/libmrb.so. Returns the library path."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        hipcc = "hipcc"
    tmp = LIB + ".tmp"
    flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    objects = [os.path.join(CSRC, src.replace(".hip", ".o")) for src in SOURCES]
    commands = [[hipcc] + flags + ["-c", "-o", obj, os.path.join(CSRC, src)] for src, obj in zip(SOURCES, objects)]
    runs = []
    for cmd in commands:  # side by side
        if verbose:
            print(" ".join(cmd), flush=True)
        runs.append(subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True))
    noise = "is not a recognized feature for this target"

    def end(run):
        text = "\n".join(line for line in run.communicate()[0].splitlines() if noise not in line)
        if run.returncode != 0:
            raise RuntimeError("hipcc failed:\n" + text)
        if verbose and text.strip():
            print(text)

    failures = []
    for run in runs:
        try:
            end(run)
        except RuntimeError as e:
            failures.append(str(e))
    if failures:
        raise RuntimeError("\n".join(failures))
    end(subprocess.Popen([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objects, stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True))
    os.replace(tmp, LIB)
    for obj in objects:
        os.remove(obj)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
    sys.exit(0)
