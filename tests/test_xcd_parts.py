"""The deal of M2L's work groups to the 8 XCDs (defmm_amd/csrc/xcd_parts.hpp),
checked on the CPU by a plain C++ program: segments, parts of equal cost, the
rotation of the parts over the chunks of right-hand sides."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_chunk_and_group_once(tmp_path):
    exe = tmp_path / "xcd_parts_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall",
                           os.path.join(ROOT, "tests", "cpp", "xcd_parts_check.cpp"),
                           "-o", str(exe)])
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    m = re.match(r"ok (\d+) cases, of one segment (\d+), two (\d+), eight (\d+)", run.stdout)
    assert run.returncode == 0 and m, run.stdout
    assert all(int(x) > 0 for x in m.groups()), run.stdout
