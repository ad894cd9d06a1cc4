"""Build recipe for libksa_hip.so (hipcc, gfx950 only) and _fast.so (the native front of the hottest calls, g++ against the
installed PyTorch)."""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libksa_hip.so")
FAST = os.path.join(HERE, "_fast.so")
# (the slowest units first: they run next to the others)
SOURCES = ["ksa_prefill_d256_bf16_regular.hip", "ksa_prefill_d256_bf16_general.hip", "ksa_prefill_d256_f16_regular.hip",
           "ksa_prefill_d256_f16_general.hip", "ksa_prefill_d256_bf16_marked.hip", "ksa_prefill_d256_f16_marked.hip",
           "ksa_prefill_d256_bf16_chunks.hip", "ksa_prefill_d256_f16_chunks.hip",
           "ksa_prefill.hip", "ksa_prefill_chunks.hip", "ksa_api.hip", "ksa_index.hip", "ksa_decode.hip", "ksa_decode_weights.hip", "ksa_cache.hip", "ksa_prompt.hip",
           "ksa_pre.hip", "ksa_elementwise.hip", "ksa_gemm_rows.hip", "ksa_mlp_rows.hip", "ksa_norm_gemm_rows.hip"]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    # scores never hold NaN unless the inputs do; without this every fmax is preceded by a
    # canonicalising v_max
    "-fno-honor-nans",
]


def _fast_command() -> list:
    import sysconfig
    import torch
    at = os.path.dirname(os.path.abspath(torch.__file__))
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"))))
    include = [os.path.join(at, "include"), os.path.join(at, "include", "torch", "csrc", "api", "include"),
               os.path.join(rocm, "include"), sysconfig.get_paths()["include"], os.path.join(os.path.dirname(HERE), "include")]
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared",
            "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",  # what the headers of ROCm and of PyTorch ask for
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(a for d in include for a in ("-isystem", d)),
            os.path.join(CSRC, "ksa_fast.cpp"), "-o", FAST, "-L" + os.path.join(at, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu",
            "-ltorch_hip", "-ltorch", "-ltorch_python", "-Wl,-rpath," + os.path.join(at, "lib")]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # the host pass warns that it does not know the packed-fp32 feature; that is expected
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"{os.path.basename(cmd[0])} failed ({res.returncode}):\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)


def _build_fast(verbose):
    try:
        _run(_fast_command(), verbose)
    except (RuntimeError, OSError) as e:
        if os.path.exists(FAST):   # of another build
            os.remove(FAST)
        print(f"_fast.so was not built, calls go through Python: {e}", file=sys.stderr)


def build(verbose: bool = False, extra_flags=(), out: str = LIB, csrc: str = CSRC, jobs: int = 8) -> str:
    """Compiles every source of `csrc` (one hipcc process each, `jobs` at a time) and links them
    into `out`.  Objects go to a `build/` folder next to `out`, named after it.  With the package's own library
    comes the native front; where that does not compile, the package does without it."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objdir = os.path.join(os.path.dirname(os.path.abspath(out)), "build",
                          os.path.splitext(os.path.basename(out))[0])
    os.makedirs(objdir, exist_ok=True)
    objs = [os.path.join(objdir, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    cmds = [[hipcc, *FLAGS, *extra_flags, "-I", csrc, "-c", os.path.join(csrc, s), "-o", o]
            for s, o in zip(SOURCES, objs)]
    with ThreadPoolExecutor(max_workers=max(1, jobs)) as pool:
        front = pool.submit(_build_fast, verbose) if out == LIB else None
        list(pool.map(lambda c: _run(c, verbose), cmds))
        if front is not None:
            front.result()
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out, *objs], verbose)
    return out


if __name__ == "__main__":
    print(build(verbose=True))
