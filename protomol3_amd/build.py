"""Builds the gfx950 engine library (libpmx.so) in-tree with hipcc."""
from __future__ import annotations

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(HERE, "lib", "libpmx.so")
SOURCES = [os.path.join(HERE, "csrc", f) for f in ("pmx.hip", "pmx_pair.hip", "pmx_pair64.hip", "pmx_pair.h",
                                                   "pmx_kernels.h", "pmx_batch.h", "pmx_common.h")]
# options of single files
FILE_FLAGS = {
    # see the head of the file
    "pmx_pair.hip": ["-mllvm", "-structurizecfg-skip-uniform-regions"],
    "pmx_pair64.hip": ["-mllvm", "-structurizecfg-skip-uniform-regions"],
}

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-munsafe-fp-atomics",
    # packed FP32 arithmetic is kept off (only scalar/FMA FP32 VALU forms)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result", "-Wno-unused-value",
]


def build_lib(verbose: bool = False) -> str:
    os.makedirs(os.path.dirname(LIB), exist_ok=True)
    jobs = []
    for src in (s for s in SOURCES if s.endswith(".hip")):
        obj = os.path.join(os.path.dirname(LIB), os.path.basename(src) + ".o")
        cmd = ["hipcc", *HIPCC_FLAGS, *FILE_FLAGS.get(os.path.basename(src), []), "-I" + os.path.join(ROOT, "include"),
               "-c", src, "-o", obj]
        jobs.append((obj, subprocess.Popen(cmd, stdout=subprocess.DEVNULL, stderr=subprocess.PIPE, text=True)))
    failed = [err for err in (p.communicate()[1] for _, p in jobs) if err and "error" in err]
    if any(p.returncode for _, p in jobs):
        raise RuntimeError("hipcc failed:\n" + "\n".join(failed)[-4000:])
    r = subprocess.run(["hipcc", "--offload-arch=gfx950", "-fPIC", "-shared", *(obj for obj, _ in jobs),
                        "-o", LIB + ".tmp"], capture_output=True, text=True)
    for obj, _ in jobs:
        os.remove(obj)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + r.stderr[-4000:])
    os.replace(LIB + ".tmp", LIB)
    if verbose:
        print("built", LIB)
    return LIB


HOST_EXE = os.path.join(HERE, "lib", "pmx_force")


def build_host(verbose: bool = False) -> str:
    """The C++ ProtoMol-boundary layer and its driver, linked to libpmx.so."""
    host = os.path.join(HERE, "host")
    cmd = ["g++", "-O2", "-std=c++17", "-Wall", "-I" + os.path.join(ROOT, "include"),
           os.path.join(host, "pmx_protomol.cpp"), os.path.join(host, "pmx_force.cpp"),
           "-L" + os.path.dirname(LIB), "-lpmx", "-Wl,-rpath,$ORIGIN", "-o", HOST_EXE + ".tmp"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed:\n" + r.stderr[-4000:])
    os.replace(HOST_EXE + ".tmp", HOST_EXE)
    if verbose:
        print("built", HOST_EXE)
    return HOST_EXE


SERVE_LIB = os.path.join(HERE, "lib", "libpmx_serve.so")


def build_serve(verbose: bool = False) -> str:
    """The request loop (host C++ over the C ABI), linked to libpmx.so."""
    cmd = ["g++", "-O2", "-std=c++17", "-Wall", "-fPIC", "-shared", "-pthread", "-I" + os.path.join(ROOT, "include"),
           os.path.join(HERE, "host", "pmx_serve.cpp"), "-L" + os.path.dirname(LIB), "-lpmx",
           "-Wl,-rpath,$ORIGIN", "-o", SERVE_LIB + ".tmp"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed:\n" + r.stderr[-4000:])
    os.replace(SERVE_LIB + ".tmp", SERVE_LIB)
    if verbose:
        print("built", SERVE_LIB)
    return SERVE_LIB


CHECK_LIB = os.path.join(ROOT, "tests", "native", "libpairfunctions.so")


def build_checks(verbose: bool = False) -> str:
    """Device functions of the pair kernel behind a C entry, for the tests."""
    src = os.path.join(ROOT, "tests", "native", "pair_functions.hip")
    r = subprocess.run(["hipcc", *HIPCC_FLAGS, "-shared", src, "-o", CHECK_LIB + ".tmp"], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + r.stderr[-4000:])
    os.replace(CHECK_LIB + ".tmp", CHECK_LIB)
    if verbose:
        print("built", CHECK_LIB)
    return CHECK_LIB


if __name__ == "__main__":
    build_lib(verbose=True)
    build_host(verbose=True)
    build_serve(verbose=True)
    build_checks(verbose=True)
