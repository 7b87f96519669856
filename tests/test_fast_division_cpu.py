"""The division by a number the launch fixes (``FastDiv`` in csrc/wave.hpp), its two formulas in Python integers
with the widths of the C++: exact for every divisor up to 2^31 - 1 and every numerator below 2^31."""
import random

import pytest


def by(d):
    shift = 0
    while shift < 31 and (1 << shift) < d:
        shift += 1
    mul = ((1 << (31 + shift)) + d - 1) // d
    assert (1 << (31 + shift)) + d - 1 < 1 << 64 and mul < 1 << 32  # what the C++ computes them in
    return mul, shift


def div(n, mul, shift):
    return ((n << 1) * mul >> 32) >> shift


LIMIT = (1 << 31) - 1
POWERS = [1 << k for k in range(31)]
DIVISORS = sorted({d for p in POWERS for d in (p - 1, p, p + 1, 3 * p) if 1 <= d <= LIMIT} | {LIMIT, LIMIT - 1, 65, 129, 1001, 46341})


@pytest.mark.parametrize("chunk", range(4))
def test_quotients_are_exact(chunk):
    rng = random.Random(chunk)
    divisors = DIVISORS[chunk::4] + [rng.randint(1, LIMIT) for _ in range(2000)] + [rng.randint(1, 5000) for _ in range(2000)]
    for d in divisors:
        mul, shift = by(d)
        top = LIMIT // d
        quotients = {0, 1, 2, top, top - 1, top // 2, rng.randint(0, top), rng.randint(0, top)}
        for n in {q * d + r for q in quotients for r in (-1, 0, 1, d - 1)} | {0, LIMIT, LIMIT - 1}:
            if 0 <= n <= LIMIT:
                assert div(n, mul, shift) == n // d, (n, d)
