"""Near-field work items (defmm_amd/csrc/near_items.hpp) on the CPU: a C++
program builds plans with the host builder, walks the items and checks that
every target meets every source of its leaf's list once, and that the check
made at upload refuses lists that leave their leaf's sources or targets."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_near_items_cover_their_lists(tmp_path):
    exe = tmp_path / "near_items_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-fopenmp", "-ffp-contract=off",
                           os.path.join(ROOT, "tests", "cpp", "near_items_check.cpp"),
                           os.path.join(ROOT, "defmm_amd", "csrc", "plan.cpp"), "-o", str(exe)])
    env = dict(os.environ, OMP_NUM_THREADS=os.environ.get("OMP_NUM_THREADS", "8"))
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300, env=env)
    print(run.stdout)
    rows = re.findall(r"^case \S+ \d+ (\S+) .* tried (\d+) missed (\d+)$", run.stdout, re.M)
    assert run.returncode == 0 and len(rows) == 8, run.stdout + run.stderr
    assert all(r == ("OK", "400", "0") for r in rows)
