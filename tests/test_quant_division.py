"""The quantizers' division by multiply-adds on the CPU, in exact rationals.

The row pass of csrc/quant_rows.h divides w by s as q = RN(w r), RN(q + RN(w - q s) r) with
r = RN(1 / s). Both operands have few mantissas: w is bf16, s is RN(amax / c) of a bf16 amax (INT8
and INT4: rounded to bf16 again) or the least scale. Every pair of them, powers of two apart, gives
the correctly rounded w / s.
"""
from __future__ import annotations

from fractions import Fraction as F

import pytest


def _round(x, bits):
    """x > 0 or < 0 rounded to ``bits`` significant bits, ties to even."""
    if x == 0:
        return x
    a = abs(x)
    e = a.numerator.bit_length() - a.denominator.bit_length()
    if F(2) ** e > a:
        e -= 1
    ulp = F(2) ** (e - bits + 1)
    n, r = divmod(a, ulp)
    if 2 * r > ulp or (2 * r == ulp and n % 2):
        n += 1
    return n * ulp if x > 0 else -n * ulp


@pytest.mark.parametrize("divisor,bf16", [(448, False), (127, True), (7, True)], ids=["fp8", "int8", "int4"])
def test_division_is_correctly_rounded(divisor, bf16):
    scales = {_round(F(a, 128) / divisor, 24) for a in range(128, 256)}
    if bf16:
        scales = {_round(s, 8) for s in scales}
    scales.add(_round(F(1, 10 ** 12), 24))
    for s in scales:
        r = _round(1 / s, 24)
        for m in range(128, 256):
            w = F(m, 128)
            q = _round(w * r, 24)
            assert _round(q + _round(w - q * s, 24) * r, 24) == _round(w / s, 24), (w, s)
