"""Builds libmctsnc_hip.so (search engine) and libpuct_hip.so (PUCT select/backup) for gfx950 with hipcc, and _puct_call
(the Python side of a PUCT launch, host code only) with the C compiler, in-tree, next to this file."""
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmctsnc_hip.so")
PUCT_LIB = os.path.join(HERE, "libpuct_hip.so")
LIBRARIES = {LIB: ["mctsnc_engine.hip"], PUCT_LIB: ["puct_kernels.hip", "puct_gomoku.hip"]}
HIPCC_FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
               # UCB values must be bit-reproducible: no fused multiply-add contraction anywhere
               "-ffp-contract=off",
               "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               # the playout loops are a few hundred bytes run by a lone wavefront: where they start relative to the
               # instruction cache lines moved measured rates by 3 % between otherwise identical builds
               "-falign-loops=64",
               "-Wno-unknown-warning-option"]
# The PUCT kernels claim with one lane of a wavefront (`if (lane == 0) atomicAdd(...)`).  The compiler's pass that turns a
# wavefront's atomics on one address into one atomic of the sum does not see that a single lane is active, and wraps
# each claim in a lane count and a broadcast (a dozen instructions per claim in kernels bound by instruction issue;
# the node-level winner-recalc selection is 4-5 % faster without it).
EXTRA_FLAGS = {PUCT_LIB: ["-mllvm", "-amdgpu-atomic-optimizer-strategy=None"]}


HOST_MODULE = os.path.join(HERE, "_puct_call" + (sysconfig.get_config_var("EXT_SUFFIX") or ".so"))


def run(cmd, what, verbose):
    if verbose:
        print(" ".join(cmd))
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"{what} failed:\n" + out)
    if verbose and out.strip():
        print(out)


def build_host_module(verbose=False, optional=False):
    """Compiles _puct_call; `optional`: where there is no C compiler or no Python.h (3.9 or later) the package does without it
    (puct.py makes the same checks in Python), and one left from an earlier build goes, since its source may have been another."""
    compiler, include = os.environ.get("CC") or "gcc", sysconfig.get_paths()["include"]
    missing = None
    if shutil.which(compiler.split()[0]) is None:
        missing = f"no C compiler ({compiler})"
    elif not os.path.exists(os.path.join(include, "Python.h")):
        missing = f"no Python.h in {include}"
    elif sys.version_info < (3, 9):
        missing = "it calls functions of Python 3.9"
    if missing and optional:
        print(f"{os.path.basename(HOST_MODULE)} is not built: {missing}; a PUCT launch on torch tensors takes a few microseconds longer", file=sys.stderr)
        if os.path.exists(HOST_MODULE):
            os.remove(HOST_MODULE)
        return None
    if missing:
        raise RuntimeError(f"{os.path.basename(HOST_MODULE)} cannot be built: {missing}")
    command = compiler.split() + ["-O2", "-Wall", "-fPIC", "-shared", "-I" + include, "-o", HOST_MODULE, os.path.join(CSRC, "puct_call.c")]
    exchange = dlpack_flags()
    try:
        run(command + exchange, "the C compiler", verbose)
    except RuntimeError:
        if not exchange:
            raise
        run(command, "the C compiler", verbose)   # (without torch's exchange table: by the tensors' attributes)
    return HOST_MODULE


def dlpack_flags():
    """Flags with which _puct_call reads tensors through the exchange table that torch publishes, where torch's DLPack header has it."""
    spec = importlib.util.find_spec("torch")
    include = os.path.join(os.path.dirname(spec.origin), "include") if spec is not None and spec.origin else ""
    header = os.path.join(include, "ATen", "dlpack.h")
    if not include or not os.path.exists(header):
        return []
    with open(header, errors="replace") as f:
        return ["-I" + include, "-DPUCT_CALL_DLPACK=<ATen/dlpack.h>"] if "DLPackExchangeAPI" in f.read() else []


def build_one(lib, sources, verbose=False):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc] + HIPCC_FLAGS + EXTRA_FLAGS.get(lib, []) + ["-o", lib] + [os.path.join(CSRC, s) for s in sources]
    run(cmd, "hipcc", verbose)
    return lib


def build(verbose=False, only=None):
    """Compiles every library (or the one whose path is `only`), and _puct_call where that can be done; returns the search engine's path."""
    for lib, sources in LIBRARIES.items():
        if only is None or only == lib:
            build_one(lib, sources, verbose)
    if only is None or only == HOST_MODULE:
        build_host_module(verbose, optional=only is None)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
