"""The host side of large transfers (threads, streams, chunks) compiled for the
CPU against a few HIP calls of its own (tests/host_hip), where calls at the same
time, other devices and failing copies can be made to happen."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("program", ["copy_lanes", "op3_chunks"])
def test_transfers_on_the_cpu(tmp_path, program):
    src, exe = os.path.join(HERE, "host_hip", program + ".cpp"), str(tmp_path / program)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", os.path.join(HERE, "host_hip"), src, "-o", exe],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout + r.stderr
