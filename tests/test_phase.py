"""The near field's table-driven cos and sin of kappa * r (defmm_amd/csrc/
phase.hpp), compiled for the CPU and checked against long double over phases
up to 1,000 radians, the midpoints between table angles and tiny distances."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_phase_table_accuracy(tmp_path):
    exe = tmp_path / "phase_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                           os.path.join(ROOT, "tests", "cpp", "phase_check.cpp"), "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300, check=True).stdout
    rows = re.findall(r"double (\S+) float (\S+) rounded_first (\S+)", out)
    assert len(rows) == 7, out
    for d, f, r in rows:
        # double: table entry and final sum rounded once each below 1 (2^-54
        # each), the correction's roundings (3 of 0.0123 * 2^-53), and the
        # long double reference's own kappa * r (1000 * 2^-64)
        assert float(d) <= 2 * 2.0 ** -54 + 3 * 0.0123 * 2.0 ** -53 + 1000 * 2.0 ** -64, out
        # float: table entry, inner and outer sum (2^-25 each), remainder
        # rounded to float (0.0123 * 2 * 2^-24), omitted y^4 / 24
        assert float(f) <= 3 * 2.0 ** -25 + 0.0123 * 2.0 ** -23 + 1e-9, out
        # never worse than rounding kappa * r first
        assert float(d) <= float(r), out
    assert "select 0 1 2 2 1 2" in out, out
