"""The transform lines of M2F and F2L (dftForward, dftInverse of
defmm_amd/csrc/dft.hpp), compiled for the CPU, for every order against the
direct sums in long double."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_dft_lines(tmp_path):
    exe = tmp_path / "dft_lines_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                           os.path.join(ROOT, "tests", "cpp", "dft_lines_check.cpp"),
                           "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120, check=True).stdout
    rows = re.findall(r"L (\d+) double (\S+) float (\S+)", out)
    assert [int(r[0]) for r in rows] == list(range(2, 11)), out
    for order, d, f in rows:
        # at most P + 3 roundings along a sum of P terms (one of each product
        # and twiddle), relative to the sum of magnitudes
        n = 2 * int(order) - 1 + 3
        assert float(d) <= n * 2.0 ** -53 and float(f) <= n * 2.0 ** -24, out
