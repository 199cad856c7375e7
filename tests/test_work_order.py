"""The order in which the workgroups of the fp32 kernels take their tiles, checked on the host (tests/work_order_check.cpp)."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "sample_efficient_gpt_amd", "csrc")


def test_every_tile_is_taken_once_and_no_xcd_idles(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path / "work_order_check")
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-Werror", "-Wno-attributes", f"-I{CSRC}",
                    os.path.join(ROOT, "tests", "work_order_check.cpp"), "-o", exe], check=True)
    proc = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert proc.returncode == 0 and "VIOLATION" not in proc.stdout, proc.stdout
