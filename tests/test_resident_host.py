"""The resident solve's host-side rules (csrc/pd_resident.h), compiled for the
CPU and run there."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "sci-solver_peridynamic_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("resident") / "resident_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I", CSRC, "-o", exe,
                    os.path.join(HERE, "resident_host.cpp")], check=True)
    return exe


@pytest.mark.parametrize("check", ["wait_limit", "scratch", "places"])
def test_rule(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
