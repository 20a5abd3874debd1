"""The trial-division screen at the edges of its stages (primes below 2^10 and
2^15, groups of eight candidates) and with pairs inside and outside the
fixed-point range (m < 2^32, |x| < 2^31) in one call, against big integers."""
import math
import random

import numpy as np
import pytest

import oracle_lib as ol
import pgap

pytestmark = pytest.mark.gpu


def product_of_primes(limit):
    sieve = bytearray([1]) * (limit + 1)
    for p in range(2, int(limit ** 0.5) + 1):
        if sieve[p]:
            sieve[p * p::p] = bytes(len(range(p * p, limit + 1, p)))
    return math.prod(p for p in range(2, limit + 1) if sieve[p])


# N that survive a stage are rare: half of the pairs are made from a survivor
@pytest.mark.parametrize("limit", [1, 2, 3, 1009, 1021, 1031, 32749, 32771, 40009, 200003])
@pytest.mark.parametrize("count", [1, 8, 9, 203])
def test_screen_matches_big_integers(engine, limit, count):
    P, D = 101, 210
    K, fam, prod, low = ol.K(P, D), engine.family(P, D, 0), product_of_primes(limit), product_of_primes(min(limit, 500))
    rng = random.Random(1000 * limit + count)
    edge_m = [1, (1 << 32) - 1, 1 << 32, (1 << 32) + 1, (1 << 63) + 5, (1 << 64) - 1]
    edge_x = [0, 1, -1, (1 << 31) - 1, 1 << 31, -(1 << 31), -(1 << 31) - 1, (1 << 62) + 3, -(1 << 62) - 3]
    pairs = []
    for i in range(count):
        m = rng.choice(edge_m) if i % 5 == 4 else rng.randrange(1, 1 << 32)
        x = rng.choice(edge_x) if i % 7 == 6 else rng.randrange(-(1 << 31), 1 << 31)
        while i % 2 and (math.gcd(abs(m * K + x), low) != 1 or math.gcd(abs(m * K + x), prod) != 1):
            x -= 1
        pairs.append((m, x))
    m = np.array([p[0] for p in pairs], dtype=np.uint64)
    x = np.array([p[1] for p in pairs], dtype=np.int64)
    keep = engine.filter_candidates(fam, m, x, limit)
    want = [int(math.gcd(abs(a * K + b), prod) == 1) for a, b in pairs]
    assert keep.tolist() == want


def test_primes_past_the_exact_window(engine):
    # above 2^28 the fixed-point window can hold a neighbouring residue, and
    # the exact one decides: multiples of primes there, and their neighbours
    P, D, limit = 101, 210, (1 << 28) + 200_000
    K, fam = ol.K(P, D), engine.family(P, D, 0)
    primes = [p for p in range((1 << 28) - 199_999, limit, 998) if ol.probab_prime(p)]
    assert sum(p > 1 << 28 for p in primes) > 5 and sum(p < 1 << 28 for p in primes) > 2
    pairs = []
    for i, p in enumerate(primes):
        m = 4_000_000_007 - 210 * i
        r = -(m * K) % p
        pairs += [(m, r), (m, r + 1), (m, r - 1), (m, r - p), (m, r - p + 1)]
    m = np.array([a for a, _ in pairs], dtype=np.uint64)
    x = np.array([b for _, b in pairs], dtype=np.int64)
    keep = engine.filter_candidates(fam, m, x, limit)
    small = engine.filter_candidates(fam, m, x, 1_000_000)
    for (a, b), k, s in zip(pairs, keep, small):
        n = a * K + b
        if any(n % p == 0 for p in primes):
            assert not k
        elif k:
            assert s
