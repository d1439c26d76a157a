"""The growth rules of a handle's workspace, adapter buffer and staging slots
(relux_amd/csrc/rlx_scratch.h) on the CPU, over an allocator that refuses on
demand: tests/scratch_host.cpp holds the scenarios."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "relux_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("scratch") / "scratch_host")
    subprocess.run(["g++", "-std=c++17", "-g", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(HERE, "scratch_host.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("scenario", ["held", "refused", "no_doubling", "last_resort", "reserved", "stage"])
def test_scratch(program, scenario):
    r = subprocess.run([program, scenario], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
