"""Builds libmrb.so (the HIP replay-buffer library) for gfx950 with hipcc, and the extension module that calls it from
Python (_native.so, host code only) with the C++ compiler, in-tree."""
import os
import subprocess
import sys
import sysconfig

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
LIB = os.path.join(CSRC, "libmrb.so")
NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_native.so")

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


SOURCES = ["mrb.hip", "mrb_push_many.hip", "mrb_range.hip", "mrb_range_one.hip", "mrb_returns.hip", "mrb_returns_streamed.hip", "mrb_sample_lanes.hip", "mrb_samples.hip", "mrb_samples_large.hip", "mrb_short.hip", "mrb_silent.hip"]


def _native_commands(tmp, obj):
    """Compiles csrc/native.cpp against torch's headers, and links it with libmrb.so (found beside it at run time)."""
    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cxx = os.environ.get("CXX", "g++")
    return ([cxx, "-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
             "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
             "-isystem", os.path.join(root, "include"), "-isystem", os.path.join(root, "include", "torch", "csrc", "api", "include"),
             "-isystem", os.path.join(rocm, "include"), "-isystem", sysconfig.get_paths()["include"],
             "-c", "-o", obj, os.path.join(CSRC, "native.cpp")],
            [cxx, "-shared", "-o", tmp, obj, "-L" + os.path.join(root, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch",
             "-ltorch_python", "-L" + CSRC, "-l:libmrb.so", "-Wl,-rpath,$ORIGIN/csrc"])


def build(verbose=False):
    """Compile the sources of mindrl_amd/csrc into mindrl_amd/csrc/libmrb.so and mindrl_amd/_native.so. Returns the path
    of the former."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    if not os.path.exists(hipcc):
        hipcc = "hipcc"
    flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    objects = [os.path.join(CSRC, src.replace(".hip", ".o")) for src in SOURCES]
    native_obj = os.path.join(CSRC, "native.o")
    compile_native, link_native = _native_commands(NATIVE + ".tmp", native_obj)
    noise = "is not a recognized feature for this target"

    def start(cmd):
        if verbose:
            print(" ".join(cmd), flush=True)
        return subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)

    def finish(runs):
        failures = []
        for run in runs:
            text = "\n".join(line for line in run.communicate()[0].splitlines() if noise not in line)
            if run.returncode != 0:
                failures.append("%s failed:\n%s" % (run.args[0], text))
            elif verbose and text.strip():
                print(text)
        if failures:
            raise RuntimeError("\n".join(failures))

    finish([start([hipcc] + flags + ["-c", "-o", obj, os.path.join(CSRC, src)]) for src, obj in zip(SOURCES, objects)]
           + [start(compile_native)])  # side by side
    finish([start([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB + ".tmp"] + objects)])
    os.replace(LIB + ".tmp", LIB)
    finish([start(link_native)])
    os.replace(NATIVE + ".tmp", NATIVE)
    for obj in objects + [native_obj]:
        os.remove(obj)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
    sys.exit(0)
