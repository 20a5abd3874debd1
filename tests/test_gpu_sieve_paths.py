"""The device sieve's two routes for large primes (64-bit fixed point while the
m's are small enough for the limit, exact residues otherwise) and its list
kernel at the edges of words and tiles, against the oracle sieve."""
import numpy as np
import pytest

import oracle_lib as ol
import pgap

pytestmark = pytest.mark.gpu

# 17 m's: two groups of eight and a remainder; the second set takes the exact route
SMALL = list(range(101, 1801, 106)) + [(1 << 20) + 1]
LARGE = [1, 1009, (1 << 31) + 11, (1 << 32) - 1, (1 << 32) + 1, (1 << 40) + 7]


@pytest.mark.parametrize("P,D,SL,limit,ms", [
    (101, 210, 1, 2, SMALL), (101, 210, 31, 64, SMALL), (101, 210, 32, 67, SMALL), (101, 210, 33, 10_000, SMALL),
    (503, 210, 8191, 300_000, SMALL), (503, 210, 8192, 300_000, LARGE), (503, 210, 8193, 2_000_000, SMALL),
    (1511, 2190, 40000, 80_001, SMALL), (1511, 2190, 40001, 5_000_000, LARGE), (13, 1, 20000, 40_013, SMALL),
])
def test_lists_match_the_oracle(engine, P, D, SL, limit, ms):
    got = engine.sieve(engine.family(P, D, SL), ms, limit, SL)
    sv = ol.Sieve(P, D, SL, limit)
    for m, (p, n) in zip(ms, got):
        wp, wn = sv(m)
        assert np.array_equal(p, wp) and np.array_equal(n, wn), m


def test_routes_agree_past_2_32(engine):
    # primes up to 4.4e9: the m's alone stay in fixed point, with a 41-bit m
    # among them the whole call takes the exact route
    SL, limit = 11000, 4_400_000_000
    fam = engine.family(907, 2190, SL)
    ms = [1, 17, 1009, 99991, 1 << 20, 7, 11, 13, 19]
    fixed = engine.sieve(fam, ms, limit, SL)
    exact = engine.sieve(fam, ms + [(1 << 40) + 7], limit, SL)
    for (p, n), (wp, wn) in zip(fixed, exact):
        assert np.array_equal(p, wp) and np.array_equal(n, wn)
