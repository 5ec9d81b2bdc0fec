"""The host's decision on the two-product quotient against trying every significand.

two_product_exact looks only at dividends whose quotients lie next to a midpoint
of two floats; here its answer is compared with the enumeration of a whole binade
for divisors of every kind: few significant bits, many, large, close to a power
of two, and the ones among 1200 random divisors that the quotient misses.
"""
from __future__ import annotations

import numpy as np
import pytest

import fs2d_amd
from test_division import binade_misses, two_product_pair

DIVISORS = [1.5, 3.0, 7.0, 1.0 + 2.0 ** -23, 2.0 - 2.0 ** -23, 1.0 + 4 * 0.8405, 1.0 + 4 * 8.405, 33.621, 1025.0, 65537.0,
            8388607.0, 16777213.0, 1.0 + 4 * 3.7e5, 2.0 ** 30 * 1.75, 1.87, 3.832235097885132, 12.917113304138184, 840.11]


@pytest.mark.parametrize("d", DIVISORS)
def test_check_agrees_with_every_significand(d):
    d32 = np.float32(d)
    y, yl = two_product_pair(d32)
    assert yl > 0
    assert fs2d_amd.division_plan(float(d32))["checked"] == (len(binade_misses(d32, y, yl, E=8)) == 0)


def test_check_of_random_divisors():
    rng = np.random.default_rng(3)
    for d in 1.0 + 4.0 * np.exp(rng.uniform(-12, 8, 12)):
        d32 = np.float32(d)
        y, yl = two_product_pair(d32)
        if yl > 0:
            assert fs2d_amd.division_plan(float(d32))["checked"] == (len(binade_misses(d32, y, yl, E=8)) == 0), float(d32)
