"""Builds libtmoe.so (the C-ABI library of include/tmoe.h) for gfx950 with hipcc.

The library is built in-tree, next to this file, so that it travels with the
source tree. `python -m` is not needed: call build() (the repository's
__graft_entry__.build() does).
"""
from __future__ import annotations

import os
import re
import shutil
import subprocess
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(ROOT, "include")
LIB = os.path.join(HERE, "libtmoe.so")

SOURCES = ["tmoe_kernels.hip", "tmoe_static.hip", "tmoe_api.cpp"]
# the measurement harness's hardware probes (include/tmoe_probe.h), a library of
# their own so that libtmoe.so holds only the layer
PROBE_SOURCES = ["tmoe_probe.hip"]
PROBE_LIB = os.path.join(HERE, "libtmoe_probe.so")
# the Python modules' host work (CPython extension over libtorch; no device code)
NATIVE_SOURCE = "tmoe_torch.cpp"
NATIVE_LIB = os.path.join(HERE, "_tmoe_native.so")
ARCH = "gfx950"

# Packed FP32 vector instructions are disabled for all device code: hipcc -O3
# would otherwise form them from ordinary float code.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-mcode-object-version=5",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the gfx950 library cannot be built")


def native_tag() -> str:
    """What _tmoe_native.so is compiled for: the version of the C ABI's header, torch's and
    Python's (_lib.native() loads no other)."""
    import torch
    with open(os.path.join(INCLUDE, "tmoe.h")) as f:
        abi = re.search(r"#define TMOE_ABI_VERSION (\d+)", f.read()).group(1)
    return f"abi {abi} torch {torch.__version__} {sysconfig.get_config_var('SOABI')}"


def native_cmd(out: str) -> list:
    """The host compiler's line for _tmoe_native.so, against the torch that runs it."""
    import torch
    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    return [os.environ.get("CXX") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
            "-Wno-unknown-pragmas", f'-DTMOE_NATIVE_TAG="{native_tag()}"',
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", INCLUDE,
            "-isystem", inc, "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"),
            "-isystem", sysconfig.get_paths()["include"], os.path.join(CSRC, NATIVE_SOURCE),
            "-o", out, "-L", lib, "-ltorch_python", "-ltorch_cpu", "-lc10"]


def build(verbose: bool = False) -> str:
    """Compiles every source (concurrently) and links libtmoe.so, libtmoe_probe.so and
    _tmoe_native.so; returns libtmoe.so's path. Where only _tmoe_native.so cannot be built
    (torch's or Python's headers missing), the others, all that callers of the C ABI need,
    are built before that is raised."""
    objdir = os.path.join(HERE, "_build")
    os.makedirs(objdir, exist_ok=True)
    cmds, groups = [], []
    for lib, sources in ((LIB, SOURCES), (PROBE_LIB, PROBE_SOURCES)):
        objs = []
        for src in sources:
            obj = os.path.join(objdir, src + ".o")
            lang = ["-x", "hip"] if src.endswith(".hip") else []
            cmds.append([hipcc(), *HIPCC_FLAGS, "-I", INCLUDE, "-I", CSRC, *lang, "-c",
                         os.path.join(CSRC, src), "-o", obj])
            objs.append(obj)
        groups.append((lib, objs))
    native_tmp = NATIVE_LIB + ".tmp"
    native_failed = None
    try:
        native = native_cmd(native_tmp)
    except Exception as e:   # no torch, or one without the headers' paths
        native_failed = f"{NATIVE_LIB}: {e}"
        native = None
    errors = _run_all(cmds + ([native] if native else []), verbose)
    if native:
        native_failed = errors.pop()
        if not native_failed:
            os.replace(native_tmp, NATIVE_LIB)
    for e in errors:
        if e:
            raise RuntimeError(e)
    for lib, objs in groups:
        tmp = lib + ".tmp"
        cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp,
               "-Wl,-rpath,/opt/rocm/lib"]
        _run(cmd, verbose)
        os.replace(tmp, lib)
    if native_failed:
        raise RuntimeError(native_failed)
    return LIB


# hipcc's host pass does not know the packed-fp32 feature and says so: harmless.
_NOISE = "'-packed-fp32-ops' is not a recognized feature"


def _run_all(cmds, verbose):
    """Runs the compile commands side by side; an error text or None for each."""
    procs = []
    for cmd in cmds:
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE,
                                            text=True)))
    errors = []
    for cmd, pr in procs:
        _, stderr = pr.communicate()
        err = "\n".join(l for l in stderr.splitlines() if _NOISE not in l)
        errors.append(f"build failed ({pr.returncode}): {' '.join(cmd)}\n{err}"
                      if pr.returncode != 0 else None)
        if pr.returncode == 0 and verbose and err.strip():
            print(err)
    return errors


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in res.stderr.splitlines() if _NOISE not in l)
    if res.returncode != 0:
        raise RuntimeError(f"build failed ({res.returncode}): {' '.join(cmd)}\n{err}")
    if verbose and err.strip():
        print(err)


if __name__ == "__main__":
    print(build(verbose=True))
