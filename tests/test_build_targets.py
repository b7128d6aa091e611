"""What the Makefile's targets ask for: the C library is built without torch, and without Python."""
import os
import subprocess

import pytest

PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mlu-ops_amd")


def plan(*args):
    """The commands a target would run if nothing were built."""
    r = subprocess.run(["make", "-n", "-B", "-C", PACKAGE] + list(args), capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    return r.stdout


@pytest.mark.parametrize("target", ["all", "lib"])
def test_the_library_needs_no_torch(target):
    out = plan(target, "PYTHON=false")
    assert "libmluops.so" in out and "-c %s/csrc/python/native.cpp" % PACKAGE not in out


def test_the_default_target_builds_the_python_module_where_torch_is():
    out = plan()
    assert "libmluops.so" in out and "csrc/python/native.cpp -o" in out
