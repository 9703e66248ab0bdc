"""The KV writer's int8 arithmetic, emulated exactly on the CPU: the division by 127, and the
rounding by a reciprocal against round_half_even of the correctly rounded quotient."""

from __future__ import annotations

from fractions import Fraction

import numpy as np
import pytest


def _round32(x: Fraction) -> np.float32:
    """The float32 nearest to x, ties to even (x positive and normal)."""
    f = np.float32(float(x))
    best = min((f, np.nextafter(f, np.float32(0)), np.nextafter(f, np.float32(np.inf))),
               key=lambda c: (abs(Fraction(float(c)) - x), int(c.view(np.uint32)) & 1))
    return np.float32(best)


def _maxima():
    """Every maximum a row can have: the fp16 magnitudes from 1e-6 on, and the floor."""
    h = np.arange(1, 0x7C00, dtype=np.uint16).view(np.float16).astype(np.float32)
    return np.concatenate([[np.float32(1e-6)], h[h > np.float32(1e-6)]])


def test_division_by_127_is_correctly_rounded_for_every_row_maximum():
    inv = np.float32(1.0) / np.float32(127.0)
    for a in _maxima():
        q = np.float32(a * inv)
        rem = _fma_exact(-q, np.float32(127.0), a)  # the remainder is a float32: no rounding
        got = _round32(Fraction(float(rem)) * Fraction(float(inv)) + Fraction(float(q)))
        assert got == np.float32(a / np.float32(127.0)), a


def _fma_exact(a, b, c) -> np.float32:
    x = Fraction(float(a)) * Fraction(float(b)) + Fraction(float(c))
    f = np.float32(float(x))
    assert Fraction(float(f)) == x
    return f


@pytest.mark.parametrize("scale_dtype", [np.float16, np.float32])
@pytest.mark.parametrize("ulp", [-1, 0, 1])
def test_reciprocal_rounding_equals_the_division_where_it_is_used(scale_dtype, ulp):
    """With a reciprocal up to one ulp off, elements that the writer does not send to the division
    (2^-14 or more from a half-integer, the row's largest quotient under 127.4) round as it does."""
    r = np.random.RandomState(7 + ulp)
    used = total = 0
    for a in r.permutation(_maxima())[:2000]:
        scale = np.float32(scale_dtype(a / np.float32(127.0)))
        if scale == 0:
            continue
        inv = np.float32(1.0) / scale
        for _ in range(abs(ulp)):
            inv = np.nextafter(inv, np.float32(np.inf if ulp > 0 else 0))
        if float(a) * float(inv) >= 127.4:
            continue
        x = (r.uniform(-1, 1, 256) * a).astype(np.float16).astype(np.float32)
        x = x[np.abs(x) <= a]
        # x * inv is exact in float64; the kernel rounds its fma to the nearest integer, half to even
        p = x.astype(np.float64) * float(inv)
        got = np.rint(p)
        keep = np.abs(p - got) < 0.5 - 2.0 ** -14
        want = np.rint((x / scale).astype(np.float32))
        assert np.array_equal(got[keep], want[keep])
        used += int(keep.sum())
        total += keep.size
    assert used > 0.99 * total
