"""Which resident kernels of a process run together, checked on the CPU by a program under
tests/cpp (built here with g++ against prism_amd/csrc/resident_ticket.h)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_resident_ticket(tmp_path):
    exe = str(tmp_path / "resident_ticket_check")
    subprocess.run(["g++", "-O2", "-std=c++20", "-pthread", os.path.join(ROOT, "tests", "cpp", "resident_ticket_check.cpp"),
                    "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr)
    assert r.returncode == 0
    assert r.stdout.strip().endswith("ok")
