"""The chunk scheduler on the CPU, over a host stand-in of the kernel layer: launches per list of
allreduces, results, and how much workspace a replay asks for."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="no g++")
def test_lists_share_launches_and_workspaces_grow_with_the_tensors(tmp_path):
    exe = str(tmp_path / "sched_host")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(ROOT, "mccl_amd", "csrc"),
                        os.path.join(HERE, "native", "sched_host.cpp"), os.path.join(HERE, "native", "null_mcclx.cpp"),
                        os.path.join(ROOT, "mccl_amd", "csrc", "mcclx_sched.cpp"), "-o", exe, "-lpthread"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout[-4000:] + r.stderr
