"""The batched kernel's Coulomb table (gomc_amd/csrc/coul_table.hpp), built and
evaluated on the CPU by the code that the kernel's set-up and the kernel run,
against erfc(alpha r) / r in extended precision over dense r^2 up to the cutoff,
row edges included.

Bar: rounding of the last multiply-add, of c0 and, times the sixth by which the
other terms can reach c0, of the rest: 4e-16; and the interpolation error of
degree 8 in a row of half width 1/128 of r^2, where ln f falls by (x^2 + 1) / 128,
x^2 = -ln(tolerance) at the cutoff: ((x^2 + 1) / 128)^9 / (2^8 9!), doubled for
the derivatives that x^2 leaves out.  Throughout it must be below 8e-15 for
tolerances down to 1e-10, what exp(-x^2) erfcx(x) with the fitted erfcx has at
1e-6.
"""
import math
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("coul") / "check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-o", str(exe),
                    str(HERE / "coul_table_check.cpp")], check=True)

    def run(tol, rcut, ewald):
        r = subprocess.run([str(exe), repr(tol), repr(rcut), str(int(ewald))],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stdout
        worst, rms, first, count = r.stdout.split()
        assert int(count) > 16 * 64 * 8
        return float(worst), float(rms), float(first)
    return run


@pytest.mark.parametrize("rcut", [4.0, 8.0, 9.7, 10.0, 11.4, 12.0, 16.0, 16.1, 23.0])
@pytest.mark.parametrize("tol", [1e-4, 1e-5, 1e-6, 1e-8, 1e-10])
def test_factor(check, tol, rcut):
    worst, rms, first = check(tol, rcut, True)
    bound = 4e-16 + 2 * ((1 - math.log(tol)) / 128) ** 9 / (2 ** 8 * math.factorial(9))
    assert worst <= bound and bound < 8e-15
    assert rms <= 2e-16
    # eight octaves, the cutoff in the last
    assert 2 ** -9 < first / rcut ** 2 <= 2 ** -7
    assert first == 2.0 ** (math.ceil(math.log2(rcut * rcut)) - 8)


def test_without_ewald(check):
    worst, _, _ = check(1e-5, 10.0, False)
    assert worst <= 4e-16
