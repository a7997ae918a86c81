"""Builds the search kernels for the CPU (tests/simt): the sources as they are, with LDS variables made variables of a workgroup's
thread and inline assembly replaced by what it does."""
import atexit
import functools
import multiprocessing
import os
import re
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
SIMT = os.path.join(HERE, "simt")
CSRC = os.path.join(os.path.dirname(HERE), "mcts_numba_cuda_amd", "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
CLANG = next((c for c in (shutil.which("clang++"), "/opt/rocm/lib/llvm/bin/clang++") if c and os.path.exists(c)), None)   # (vector types are clang's)

REWRITES = [
    (r"extern __shared__ (?:__attribute__\(\(aligned\(16\)\)\) )?(\w+) s_dyn\[\];", r"\1 *const s_dyn = static_cast<\1 *>(simt::dynamic_lds());"),
    (r"__shared__ ", "static thread_local "),
    (r"__attribute__\(\(address_space\(1\)\)\) ?", ""),
    (r"__attribute__\(\(amdgpu_waves_per_eu\([0-9, ]*\)\)\)", ""),
    (r'asm volatile\("s_waitcnt vmcnt\(0\)" ::: "memory"\);', ";"),
    (r'asm volatile\("" ::: "memory"\);', "simt::together_only();"),   # (the lanes are in step wherever this stands)
    (r'asm\("v_mad_u32_u24 %0, %1, %2, %3" : "=v"\((\w+)\) : "v"\((\w+)\), "s"\((\w+)\), "v"\((\w+)\)\);', r"\1 = simt::mad24(\2, (uint32_t)\3, \4);"),
    (r'asm\("v_lshlrev_b64 %0, 14, %1" : "=v"\((\w+)\) : "v"\((\w+)\)\);', r"\1 = \2 << 14;"),
    (r'asm(?: volatile)?\("" : [^;]*\);', ";"),
    (r"if \(xcd_local\) wait_own_stores_at_l2\(\);", "simt::together_only();"),   # (a store of all lanes before one of the first)
    # (one lane reads others' registers: all lanes take part)
    (r"if \(lane == 0\) \{(\n +LeafInfo li;\n)", r"{\1"), (r"\n( +)s_leaf = li;\n", r"\n\1if (lane == 0) s_leaf = li;\n"),
]

# One draw in 2^12 is rounded up to 1.0f instead of one in 2^25, in the kernels and in an oracle of its own.
FREQUENT = [
    (r"return \(float\)\(\(double\)\((mo_)?rng_next\((s0, s1|s)\) >> 11\)", r"const uint64_t x = \1rng_next(\2); if (x >> 52 == 0xfffu) return 1.0f; return (float)((double)(x >> 11)"),
    (r"( +const double d = __builtin_fma\(\(double\)hi)", r"    if (hi >> 20 == 0xfffu) return 0x1p64f;\n\1"),
    (r"( +const uint32_t rest = \(uint32_t\)output >> 11;)", r"    if (output >> 52 == 0xfffu) return 0x1p32f;\n\1"),
    (r"( +return \(uint64_t\)\(uint32_t\)\(output >> 32\) \* count)", r"    if (output >> 52 == 0xfffu) return 0;\n\1"),
]


def rewritten(text, rewrites=REWRITES, counts=None):
    """`counts`: how often each pattern has matched, added up."""
    for i, (pattern, to) in enumerate(rewrites):
        text, matches = re.subn(pattern, to, text)
        if counts is not None:
            counts[i] += matches
    assert rewrites is not REWRITES or "asm(" not in text and "asm volatile" not in text and "__shared__" not in text, re.findall(r".*(?:\basm\b|__shared__).*", text)
    return text


def folder_for_this_run():
    folder = tempfile.mkdtemp()
    atexit.register(shutil.rmtree, folder, True)
    return folder


def run(command):
    res = subprocess.run(command, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, " ".join(command) + "\n" + res.stdout[-6000:]


def build_oracle(folder):
    """The oracle with draws as in build(frequent=True)."""
    source, lib = os.path.join(folder, "oracle.c"), os.path.join(folder, "liboracle.so")
    with open(os.path.join(os.path.dirname(HERE), "oracle", "mctsnc_oracle.c")) as f, open(source, "w") as out:
        counts = [0]
        out.write(rewritten(f.read(), FREQUENT[:1], counts))
    assert all(counts), "the oracle's draws are not rounded up"
    run(["gcc", "-O2", "-std=gnu99", "-fPIC", "-fopenmp", "-ffp-contract=off", "-shared", "-o", lib, source, "-lm"])
    return lib


def build(source, folder, flags=(), libraries=(), frequent=False):
    """Compiles tests/simt/<source>.cpp and returns the shared library's path (`flags`: sanitizers, for the kernels alone;
    `frequent`: with FREQUENT draws)."""
    counts = [0] * len(FREQUENT)
    for name in os.listdir(CSRC):
        if name.endswith((".h", ".hpp")):
            with open(os.path.join(CSRC, name)) as f, open(os.path.join(folder, name), "w") as out:
                text = rewritten(f.read())
                out.write(rewritten(text, FREQUENT, counts) if frequent else text)
    assert not frequent or all(counts), [pattern for (pattern, _), n in zip(FREQUENT, counts) if n == 0]
    with open(os.path.join(CSRC, "mctsnc_engine.hip")) as f:
        engine = f.read()
    words, layout = re.search(r"^int gomoku_words\(.*?^}", engine, re.M | re.S), re.search(r"^struct GomokuLayout .*?^}", engine, re.M | re.S)
    with open(os.path.join(folder, "layout.inc"), "w") as f:
        f.write(words.group(0) + "\n" + layout.group(0) + "\n")
    lib = os.path.join(folder, f"lib{source}.so")
    common = [CLANG, "-std=c++17", "-O1", "-g", "-fPIC", "-ffp-contract=off", "-Wno-unknown-attributes", "-Wno-ignored-attributes", "-I" + folder, "-I" + SIMT, "-I" + INCLUDE]
    run(common + ["-c", "-o", os.path.join(folder, "simt.o"), os.path.join(SIMT, "simt.cpp")])
    run(common + list(flags) + ["-c", "-o", os.path.join(folder, source + ".o"), os.path.join(SIMT, source + ".cpp")])
    run([CLANG, "-shared", "-o", lib, os.path.join(folder, "simt.o"), os.path.join(folder, source + ".o"), "-lpthread"] + list(libraries))
    return lib


CHECKED = ["-fsanitize=undefined", "-fno-sanitize=function,vptr,alignment", "-fsanitize-trap=undefined"]   # (traps: nothing to link)


@functools.lru_cache(None)
def checked(source):
    """The library of tests/simt/<source>.cpp with FREQUENT draws that ends at undefined behaviour (an index beyond an array's bounds
    among it), and the oracle that goes with it."""
    folder = folder_for_this_run()
    return build(source, folder, CHECKED, frequent=True), build_oracle(folder)


def _child(function, library, oracle, args, kw):
    from oracle import oracle as module
    module._LIB_PATH = oracle
    function(library, *args, **kw)


def run_apart(function, libraries, *args, **kw):
    """function(library, ...) in a process of its own: what the kernels' bounds end, ends that."""
    child = multiprocessing.get_context("spawn").Process(target=_child, args=(function, *libraries, args, kw))
    child.start()
    child.join(300)
    if child.is_alive():
        child.kill()
        child.join()
        raise AssertionError("has not ended")
    assert child.exitcode == 0, f"exit code {child.exitcode}"


@functools.lru_cache(None)
def thread_sanitizer():
    """ThreadSanitizer's runtime library, or None where there is none or it does not run."""
    path = CLANG and subprocess.run([CLANG, "-print-file-name=libclang_rt.tsan-x86_64.so"], stdout=subprocess.PIPE, text=True).stdout.strip()
    if not path or not os.path.isabs(path) or not os.path.exists(path):
        return None
    tried = subprocess.run([sys.executable, "-c", "pass"], env=dict(os.environ, LD_PRELOAD=path), stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    return path if tried.returncode == 0 else None


def races(source, module, cases, known=""):
    """What ThreadSanitizer has to say about module.compare(library, *case, **last of case) of the cases, in a process of its own: a
    wavefront is one thread to it, barriers and what is published between workgroups order them.  known: a function to pass over."""
    folder = folder_for_this_run()
    lib = build(source, folder, ["-fsanitize=thread", "-mllvm", "-tsan-instrument-func-entry-exit=0"], ["-fsanitize=thread", "-shared-libsan"])
    passed_over = os.path.join(folder, "known")
    with open(passed_over, "w") as f:
        f.write(f"race:{known}\n" if known else "")
    env = dict(os.environ, LD_PRELOAD=thread_sanitizer(), TSAN_OPTIONS=f"exitcode=66 suppressions={passed_over}", OMP_NUM_THREADS="1")
    code = f"import sys; sys.path[:0] = {[os.path.dirname(HERE), HERE]!r}; import {module} as t\nfor c in {cases!r}: t.compare({lib!r}, *c[:-1], **c[-1])"
    res = subprocess.run([sys.executable, "-c", code], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=600)
    return res.returncode, res.stdout
