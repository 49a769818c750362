"""Builds and runs tests/host_lists.cpp: the launch lists' host arithmetic (no
GPU needed)."""
import os
import subprocess

import pytest

from quantit_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_host_lists(tmp_path):
    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    exe = tmp_path / "host_lists"
    res = subprocess.run([cc, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-I", str(build.CSRC),
                          os.path.join(HERE, "host_lists.cpp"), "-o", str(exe),
                          "-L", str(build.PKG), "-lquantit_amd", f"-Wl,-rpath,{build.PKG}"],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout + res.stderr
