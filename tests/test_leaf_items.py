"""P2M work items (defmm_amd/csrc/leaf_items.hpp) on the CPU: a C++ program
builds plans with the host builder, among them plans whose source leaves have
no direction slots (their cells take part in no M2L), and checks that no item
starts beyond its leaf's slots and that every slot is covered once."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_p2m_items_lie_within_their_leaves_slots(tmp_path):
    exe = tmp_path / "leaf_items_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-fopenmp", "-ffp-contract=off",
                           os.path.join(ROOT, "tests", "cpp", "leaf_items_check.cpp"),
                           os.path.join(ROOT, "defmm_amd", "csrc", "plan.cpp"), "-o", str(exe)])
    env = dict(os.environ, OMP_NUM_THREADS=os.environ.get("OMP_NUM_THREADS", "8"))
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300, env=env)
    print(run.stdout)
    rows = re.findall(r"^case (\S+) (\S+) leaves (\d+) without (\d+) .* few (\d+) slots (\d+) "
                      r"mfma (\d+) big (\d+)$", run.stdout, re.M)
    assert run.returncode == 0 and len(rows) == 7, run.stdout + run.stderr
    assert all(r[1] == "OK" for r in rows)
    # the cases hold what they are meant to: leaves without slots below and
    # above the line of 2,048 leaves, and every kind of list
    assert any(int(r[2]) < 2048 and int(r[3]) for r in rows)
    assert any(int(r[2]) >= 2048 and int(r[3]) for r in rows)
    for k in range(4, 8):
        assert any(int(r[k]) for r in rows), k
