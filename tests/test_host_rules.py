"""CPU checks of the library's host rules that need no device: the headers of
csrc without HIP types, compiled for the host (tests/cxx/host_rules.cpp)."""

import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "ccpi-reconstruction_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_rules") / "host_rules")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC,
                    os.path.join(HERE, "cxx", "host_rules.cpp"), "-o", out], check=True)
    return out


@pytest.mark.parametrize("check", ["grids", "kept", "kept_threads", "refused_allocation",
                                   "cone_tiles", "par_columns", "bp_blocks", "batch_tune"])
def test_host_rule(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
