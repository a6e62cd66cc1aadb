"""Generates erfcx_poly.hpp: the polynomial of the FP64 erfc in the
whole-box forces and virial and in the device move loop, erfc(x) = exp(-x^2) * erfcx(x) for 0 <= x <= 4.

erfcx(x) = exp(x^2) erfc(x) is smooth; it is sampled at 6000 Chebyshev
nodes of [0, 4.1] (scipy.special.erfcx as the reference values), fitted by a
degree-28 Chebyshev series in least squares, and the series is converted to
monomials in t = (x - 2.05) / 2.05 for Horner evaluation; the kernel uses it
for 0 <= x <= 4.  Max relative error of exp(-x^2) times the Horner form in
double precision over [0, 4]: about 3e-15 (checked by
tests/test_erfc_poly.py against scipy.special.erfc).

Run: python gomc_amd/csrc/gen_erfcx.py  (rewrites erfcx_poly.hpp beside it)
"""
from pathlib import Path

import numpy as np
from numpy.polynomial import chebyshev as Ch
from scipy.special import erfcx

DEG, NODES, LO, HI, USE = 28, 6000, 0.0, 4.1, 4.0


def coefficients() -> np.ndarray:
    mid, half = (LO + HI) / 2, (HI - LO) / 2
    t = np.cos(np.pi * (np.arange(NODES) + 0.5) / NODES)
    c = Ch.chebfit(t, erfcx(t * half + mid), DEG)
    return Ch.cheb2poly(c)


def main() -> None:
    m = coefficients()
    lines = ",\n".join(f"    {v:.17e}" for v in m)
    out = f"""// Generated by gen_erfcx.py: monomial coefficients (ascending powers of
// t = (x - mid) / half) of a degree-{DEG} least-squares Chebyshev fit of
// erfcx(x) = exp(x^2) erfc(x) on [{LO}, {HI}], used for 0 <= x <= {USE}.
#pragma once

namespace gomc {{
constexpr int kErfcxDeg = {DEG};
constexpr double kErfcxMid = {(LO + HI) / 2!r}, kErfcxInvHalf = {2 / (HI - LO)!r};
constexpr double kErfcxUse = {USE};
__device__ constexpr double kErfcxPoly[kErfcxDeg + 1] = {{
{lines}}};
}}  // namespace gomc
"""
    Path(__file__).with_name("erfcx_poly.hpp").write_text(out)


if __name__ == "__main__":
    main()
