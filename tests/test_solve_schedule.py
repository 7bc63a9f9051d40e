"""The launch schedules of the wide triangular solves, which are plain host
code: a small C++ program (tests/native/solve_schedule_check.cpp) compiled
against the library's header walks them."""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_solve_schedules_hold_every_workgroup_once(tmp_path):
    exe = tmp_path / "check"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", str(ROOT / "probit_amd/csrc"),
                    str(ROOT / "tests/native/solve_schedule_check.cpp"), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
