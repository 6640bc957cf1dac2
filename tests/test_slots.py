"""The record slots of the binning (gpu_recip_amd/csrc/pme_slots.hpp), host code only:
slots beyond 2^31, which 2^28 atoms and more have, survive the list in which the
spread reorders its records; compiled with g++ and run on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "gpu_recip_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_slots_beyond_32_bits(tmp_path):
    exe = tmp_path / "slots_check"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC, os.path.join(HERE, "cpp", "slots_check.cpp"),
                    "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
