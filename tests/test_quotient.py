"""Known-divisor quotients of the fp64 collision (lbm_amd/csrc/quotient.hpp):
the same bits as the host's division, for the collision's constant divisors
and for relaxation times over the accepted range, on random numerators over
500 binades and on numerators next to rounding boundaries of the quotient.
No tolerance: the form is correctly rounded."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]


def test_quotient_equals_division(tmp_path):
    exe = tmp_path / "quotient_probe"
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'lbm_amd' / 'csrc'}", str(ROOT / "tests" / "quotient_probe.cpp"), "-o", str(exe)],
                   check=True)
    done, bad = map(int, subprocess.run([str(exe), "20000"], check=True, capture_output=True, text=True).stdout.split())
    assert done > 4_000_000 and bad == 0
