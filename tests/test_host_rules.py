"""Dispatch rules and workspace sizes of the library's host code (tests/cpp/host_rules.cpp), without a GPU."""
import os
import subprocess

import pytest

import __graft_entry__ as entry

EXE = os.path.join(entry.ROOT, "tests", "cpp", "bin", "host_rules")


@pytest.mark.parametrize("check", ["fit_limit"])
def test_host_rules(check):
    assert os.path.exists(EXE), "build the test programs first (python __graft_entry__.py)"
    p = subprocess.run([EXE, check], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0, p.stdout + p.stderr
