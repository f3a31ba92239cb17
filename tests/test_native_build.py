"""_tmoe_native.so is compiled against one torch: another build of it is refused, and its
failure to build does not take the C ABI's libraries with it."""
import importlib.util
import os
import stat

import pytest
import torch

from conftest import ROOT


def test_native_matches_this_torch(pkg, monkeypatch):
    lib = pkg._lib
    mod = lib.native()
    assert torch.__version__ in mod.built_for and f"abi {lib.ABI_VERSION} " in mod.built_for
    monkeypatch.setattr(lib, "_native", None)
    with monkeypatch.context() as m:
        m.setattr(torch, "__version__", "2.9.1")
        with pytest.raises(RuntimeError, match="built for"):
            lib.native()
    with monkeypatch.context() as m:
        m.setattr(lib, "ABI_VERSION", lib.ABI_VERSION + 1)
        with pytest.raises(RuntimeError, match="built for"):
            lib.native()
    assert lib._native is None and lib.native() is not None


def test_unloadable_native_is_named(pkg, monkeypatch, tmp_path):
    bad = tmp_path / "_tmoe_native.so"
    bad.write_bytes(b"not a library")
    monkeypatch.setattr(pkg._lib, "_native", None)
    monkeypatch.setattr(pkg._lib, "NATIVE_PATH", str(bad))
    with pytest.raises(RuntimeError, match="does not load"):
        pkg._lib.native()


@pytest.mark.parametrize("broken", ["headers", "torch", "kernels", None])
def test_build_without_native(monkeypatch, tmp_path, broken):
    """The build with a stand-in for both compilers: without torch's headers, or without
    torch, libtmoe.so and the probes are there when the error is raised."""
    cc = tmp_path / "cc"
    cc.write_text("#!/bin/sh\nwhile [ $# -gt 0 ]; do case $1 in -o) out=$2;; "
                  "*tmoe_torch.cpp) t=1;; *tmoe_kernels.hip) k=1;; esac; shift; done\n"
                  f"[ '{broken}' = headers ] && [ \"$t\" ] && exit 1\n"
                  f"[ '{broken}' = kernels ] && [ \"$k\" ] && exit 1\n: > $out\n")
    cc.chmod(cc.stat().st_mode | stat.S_IXUSR)
    spec = importlib.util.spec_from_file_location(
        "_tmoe_build_test", os.path.join(ROOT, "mamba-tuckermoe_amd", "_build.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    monkeypatch.setenv("CXX", str(cc))
    monkeypatch.setattr(b, "hipcc", lambda: str(cc))
    for name in ("HERE", "LIB", "PROBE_LIB", "NATIVE_LIB"):
        monkeypatch.setattr(b, name, str(tmp_path / os.path.basename(getattr(b, name)))
                            if name != "HERE" else str(tmp_path))
    if broken == "torch":
        def no_torch(out):
            raise ImportError("No module named 'torch'")
        monkeypatch.setattr(b, "native_cmd", no_torch)
    if broken:
        with pytest.raises(RuntimeError):
            b.build()
    else:
        assert b.build() == b.LIB
    assert [os.path.exists(f) for f in (b.LIB, b.PROBE_LIB, b.NATIVE_LIB)] == {
        "headers": [True, True, False], "torch": [True, True, False],
        "kernels": [False, False, True], None: [True, True, True]}[broken]
