"""Rounding of L2P's float sums on the matrix cores, modelled on the CPU with
the kernel's rule for their chains (defmm_amd/csrc/leaf_items.hpp): no larger
than the vector kernel's nested sums, apart from the one rounding more of the
product of three weights (2^-24 / sqrt(3) of a term, independent)."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_chains_round_no_worse_than_nested_sums(tmp_path):
    exe = tmp_path / "l2p_chain_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                           os.path.join(ROOT, "tests", "cpp", "l2p_chain_check.cpp"),
                           "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300, check=True).stdout
    rows = re.findall(r"order (\d+) nested (\S+) chains (\S+)", out)
    assert len(rows) == 9, out
    for L, nested, chains in rows:
        assert float(chains) <= (float(nested) ** 2 + 2.0 ** -48 / 3) ** 0.5, out
