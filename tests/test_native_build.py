"""The parts that the build makes, and that they are made for each other."""
import os
import re
import shutil
import subprocess
import sys

import pytest

from pytorch_block_sparse_amd import native

CSRC = os.path.dirname(native.LIB_PATH)
HEADER = os.path.join(os.path.dirname(os.path.dirname(CSRC)), "include", "pbs_hip.h")


def test_make_builds_what_the_package_loads():
    plan = subprocess.run(["make", "-n", "-B", "-C", CSRC], capture_output=True, text=True, check=True).stdout
    assert "-o libpbs_hip.so" in plan and "-o libpbs_hip_check.so" in plan and "build.py --torch-only" in plan
    assert "-packed-fp32-ops" in plan


def test_make_knows_every_header():
    """A change to any header that the library is made of makes the library old."""
    rules = subprocess.run(["make", "-npq", "-C", CSRC], capture_output=True, text=True).stdout
    included, seen = ["pbs_hip.hip"], set()
    while included:
        path = os.path.normpath(os.path.join(CSRC, included.pop()))
        if path in seen:
            continue
        seen.add(path)
        with open(path) as f:
            included += [os.path.join(os.path.dirname(path), name) for name in re.findall(r'^#include "(.*)"', f.read(), re.M)]
    for library in ("libpbs_hip.so", "libpbs_hip_check.so"):
        needs = re.search(r"^%s: (.*)$" % re.escape(library), rules, re.M).group(1).split()
        assert seen <= {os.path.normpath(os.path.join(CSRC, n)) for n in needs}, library


def test_version_of_the_header():
    with open(HEADER) as f:
        assert int(re.search(r"#define PBS_ABI_VERSION (\d+)", f.read()).group(1)) == native.ABI_VERSION
    assert native.load().pbs_abi_version() == native.ABI_VERSION


@pytest.mark.parametrize("version, works", [(native.ABI_VERSION, True), (native.ABI_VERSION - 1, False)])
def test_module_refuses_another_library(tmp_path, version, works):
    """_pbs_torch.so next to a library of the same exports that reports a version."""
    native.torch_path()   # (built)
    shutil.copy(os.path.join(CSRC, "_pbs_torch.so"), tmp_path)
    source = "".join('extern "C" int %s() { return %d; }\n' % (s, version) for s in native.EXPORTED_SYMBOLS)
    (tmp_path / "stub.cpp").write_text(source)
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(tmp_path / "libpbs_hip.so"), str(tmp_path / "stub.cpp")], check=True)
    code = "import sys, torch; sys.path.insert(0, %r); import _pbs_torch; print('loaded')" % str(tmp_path)
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=tmp_path)
    assert ("loaded" in run.stdout) == works, run.stderr
    assert works or "ImportError: _pbs_torch.so was built for version" in run.stderr
