"""The prefill work lists (relux_amd/csrc/rlx_prefill_plan.h) on the CPU: every
query tile's key blocks once, the parts' slots and merge entries, and where the
items run (tests/prefill_plan_host.cpp)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "relux_amd", "csrc")


def test_prefill_plan(tmp_path):
    exe = str(tmp_path / "prefill_plan_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC,
                    os.path.join(HERE, "prefill_plan_host.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert r.returncode == 0, r.stdout
