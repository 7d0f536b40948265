"""The device-memory list of a context (wbpr_amd/csrc/dev_pool.h) against a stand-in for hipMalloc: what it
holds beyond the arrays in use stays within its limit, and never makes another context's allocation fail."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

HERE = os.path.join(ROOT, "tests", "host_sanitize")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_dev_pool(tmp_path):
    exe = tmp_path / "dev_pool"
    build = subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-D_GLIBCXX_ASSERTIONS", "-pthread",
                            "-I", os.path.join(HERE, "hip_stub"),
                            os.path.join(HERE, "dev_pool_driver.cpp"), "-o", str(exe)],
                           capture_output=True, text=True, timeout=300)
    assert build.returncode == 0, build.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
