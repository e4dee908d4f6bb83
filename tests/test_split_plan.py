"""CPU test of the split-KV plans: split_plan_check.cpp, compiled here against the header
that the library's host code and its schedule kernel use."""

from __future__ import annotations

import shutil
import subprocess

import pytest

from conftest import REPO


def test_plans_fit_their_launch(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = tmp_path / "split_plan_check"
    subprocess.run([cxx, "-std=c++17", "-O2", "-o", str(exe), str(REPO / "tests" / "split_plan_check.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
