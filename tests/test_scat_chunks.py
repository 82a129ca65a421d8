"""The split of the scattered field's sources into chunks (spk_scat.h), built as
a host program: every source in one chunk, the chunks' sums in the workspace,
and no wave walking through 64 sources where the whole call has too few
workgroups to fill the chip (a 176-edge surface took 70 us for 53)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "specklesim_amd", "csrc")


def test_chunks(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ not found")
    exe = str(tmp_path / "scat_chunk_check")
    subprocess.run([cxx, "-O1", "-std=c++17", "-I", CSRC, os.path.join(HERE, "scat_chunk_check.cpp"),
                    "-o", exe], check=True, capture_output=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and "bad 0" in out.stdout, out.stdout + out.stderr
