"""Root-mean-square error of the float near field's cos and sin of kappa * r
(defmm_amd/csrc/phase.hpp), compiled for the CPU: no larger than that of
polynomials of the reduced phase, for which largest errors alone do not speak
(three roundings near 1 in a row stay below the same largest error with 1.45
times the mean)."""
import os
import re
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_float_phase_rms(tmp_path):
    exe = tmp_path / "phase_rms_check"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-ffp-contract=off",
                           os.path.join(ROOT, "tests", "cpp", "phase_rms_check.cpp"),
                           "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300, check=True).stdout
    rows = re.findall(r"table (\S+) polynomials (\S+)", out)
    assert len(rows) == 4, out
    far, shift = re.search(r"entries (\S+) shift (\S+)", out).groups()
    # 2^-29 by construction, and the shift's rounding to float (3e-4 * 2^-24)
    assert float(far) <= 2.0 ** -29 + 3e-4 * 2.0 ** -24, out
    assert float(shift) <= 3e-4, out
    for t, p in rows:
        assert float(t) <= float(p), out
        # one rounding to float of each of cos and sin, uniform within half a
        # unit of the last place, at most 2^-25: 2^-25 sqrt(2 / 3); and the
        # remainder's rounding, 0.0123 * 2^-24
        assert float(t) <= 2.0 ** -25 * (2 / 3) ** 0.5 + 0.0123 * 2.0 ** -24, out
