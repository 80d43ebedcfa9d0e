"""Build liblumx.so (HIP kernels + host runtime + C ABI) in-tree for gfx950.

Run as ``python -m lum_amd.build``; ``__graft_entry__.build()`` calls
``build()``.  Every source is compiled by hipcc in one invocation, with FMA
contraction off (the parity contract of the kernels), packed-FP32
instructions disabled, and LLVM's max-ILP machine scheduler for the GPU code
(measured 1-2% faster on every workload than the default schedule, with the
same results: scheduling does not change the arithmetic).
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "liblumx.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = ["radiance.hip", "map.hip", "glossy.hip", "probes.hip", "diffuse.hip", "blockify.hip", "residency.hip", "host.cpp", "batch.cpp", "server.cpp", "clum.cpp", "vox.cpp"]

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-mllvm", "-amdgpu-sched-strategy=max-ilp",
    "-I", os.path.join(ROOT, "include"),
]


def _compile(srcs, out: str, verbose: bool) -> str:
    tmp = out + ".tmp"
    cmd = [HIPCC] + FLAGS + ["-x", "hip"] + srcs + ["-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("hipcc failed building " + os.path.basename(out))
    os.replace(tmp, out)
    return out


def build(verbose: bool = False) -> str:
    return _compile([os.path.join(CSRC, s) for s in SOURCES], OUT, verbose)


def build_tests(verbose: bool = False) -> str:
    """tests/libmarch_device.so: the kernels' arithmetic over arrays, for the
    GPU tests that compare it with IEEE arithmetic."""
    tests = os.path.join(ROOT, "tests")
    return _compile([os.path.join(tests, "march_device.hip")], os.path.join(tests, "libmarch_device.so"), verbose)


if __name__ == "__main__":
    print(build(verbose=True))
