"""The makefile's targets on a machine whose Python has no torch, which a host of the C ABI alone may be. (The compilers are stand-ins: what
is built, and what is not asked for, is the matter here.)"""
import os
import shutil
import subprocess
import sys

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spikingbrain-7b_amd", "csrc")


@pytest.fixture
def make(tmp_path):
    csrc = tmp_path / "package" / "csrc"
    shutil.copytree(CSRC, csrc, ignore=shutil.ignore_patterns("build"))
    shutil.copytree(os.path.join(CSRC, "..", "..", "include"), tmp_path / "include")
    fake = tmp_path / "compiler"                                           # writes the file behind -o
    fake.write_text("#!/bin/sh\necho \"$@\" >> " + str(tmp_path / "compiled") + "\nwhile [ $# -gt 1 ]; do [ \"$1\" = -o ] && out=$2; shift; done\n"
                    "touch ${out:-build/$(basename $1 .hip).o}\n")
    fake.chmod(0o755)

    def run(target, python):
        env = dict(os.environ, MAKEFLAGS="")
        return subprocess.run(["make", "-C", str(csrc), target, f"HIPCC={fake}", f"CXX={fake}", f"PY={python}"], env=env, capture_output=True, text=True)
    run.package, run.compiled = tmp_path / "package", tmp_path / "compiled"
    return run


def test_without_torch(make):
    none = "/bin/false"
    first = make("lib", none)
    assert first.returncode == 0 and (make.package / "libsbcache.so").exists()
    both = make("all", none)
    assert both.returncode == 0 and "_calls.so" in both.stdout and not (make.package / "_calls.so").exists()
    only = make("calls", none)
    assert only.returncode != 0 and "no torch" in only.stderr
    assert make("clean", none).returncode == 0 and not (make.package / "libsbcache.so").exists()


def test_with_torch(make):
    done = make("all", sys.executable)
    assert done.returncode == 0 and (make.package / "_calls.so").exists()
    line = [x for x in make.compiled.read_text().splitlines() if "calls.cpp" in x]
    import torch
    flags = (make.package / "csrc" / "build" / "torch_flags").read_text()
    assert len(line) == 1 and "@build/torch_flags" in line[0] and f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}" in flags
    make("all", sys.executable)                                            # nothing changed: nothing compiled
    assert len([x for x in make.compiled.read_text().splitlines() if "calls.cpp" in x]) == 1
