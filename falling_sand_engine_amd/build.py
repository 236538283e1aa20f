"""Build libfsg.so (HIP kernels + C-ABI) for gfx950 in-tree.

Run as ``python -m falling_sand_engine_amd.build`` or through
``__graft_entry__.build()``.  The library lands in
``falling_sand_engine_amd/lib/libfsg.so``; nothing is installed elsewhere.
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libfsg.so")

SOURCES = ["fsg_kernels.hip", "fsg_api.hip", "fsg_serve.hip", "fsg_render.hip", "fsg_island.hip", "fsg_generate.hip", "fsg_pack.hip", "fsg_mesh.hip", "fsg_particles.hip", "fsg_noalloc.hip", "fsg_host.cpp"]
HEADERS = ["fsg_device.hpp", "fsg_kernels.hpp", "fsg_internal.hpp", "fsg_generate.hpp", "fsg_lz4.hpp", "fsg_lz4_wide.hpp"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("FSG_ARCH", "gfx950")

# Packed fp32 instructions are disabled for all device code.
FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "-shared", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
    "-I", os.path.join(ROOT, "include"), "-I", CSRC,
]


def build(verbose: bool = True) -> str:
    os.makedirs(LIBDIR, exist_ok=True)
    tmp = LIB + ".tmp"
    cmd = [HIPCC] + FLAGS + [os.path.join(CSRC, s) for s in SOURCES] + ["-o", tmp]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    os.replace(tmp, LIB)
    return LIB


def build_cpp_tests(verbose: bool = True) -> str:
    """The C++ facade test program (tests/cpp), linked against libfsg.so."""
    src = os.path.join(ROOT, "tests", "cpp", "world_facade_test.cpp")
    outdir = os.path.join(ROOT, "tests", "cpp", "build")
    os.makedirs(outdir, exist_ok=True)
    out = os.path.join(outdir, "world_facade_test")
    cmd = ["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "include"), src, "-L", LIBDIR, "-lfsg",
           "-Wl,-rpath,$ORIGIN/../../../falling_sand_engine_amd/lib", "-o", out]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    # the LZ4 block decoders of the device codec, built for the host
    srcs = [os.path.join(ROOT, "tests", "cpp", f) for f in ("lz4_host.cpp", "lz4_wide_host.cpp")]
    lz4 = os.path.join(outdir, "liblz4host.so")
    cmd = [HIPCC, "--offload-host-only", "-x", "hip", "-O2", "-std=c++17", "-fPIC", "-shared", "-I", CSRC] + srcs + [
        "-o", lz4]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    return out


if __name__ == "__main__":
    build(verbose="-q" not in sys.argv)
    build_cpp_tests(verbose="-q" not in sys.argv)
