"""The screen's exact check where the fixed-point window holds neighbouring
residues: for primes above 2^32 / 5 the residue 1 lies inside it and above 2^30 the
residue p - 1 too, so N = 1 or -1 (mod p) passes the window and only the exact
residue keeps it."""
import random

import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu

LIMIT = 1_200_000_000
WINDOW_TOP, MARGIN = 8, 1 << 34  # family.hip, fixed_high: high word of residue 2^64 / p + margin


def next_prime(n):
    while not ol.probab_prime(n):
        n += 1
    return n


def in_window(residue, p):
    return ((residue * (1 << 64) // p + MARGIN) % (1 << 64)) >> 32 <= WINDOW_TOP


def test_neighbours_of_large_primes_are_kept(engine):
    P, D = 101, 210
    K, fam = ol.K(P, D), engine.family(P, D, 0)
    rng = random.Random(2)
    kept, dropped = [], []
    for i, at in enumerate([870_000_000, 900_000_000, 1_000_000_000, 1_080_000_000, 1_150_000_000, 1_199_000_000]):
        p = next_prime(at)
        assert p < LIMIT
        for r in ((1, p - 1) if p > 1 << 30 else (1,)):
            assert in_window(r, p)
            for below in (False, True):
                while True:  # a prime N = r (mod p): no factor up to the limit
                    m = rng.randrange(1 << 31, 1 << 32)
                    x = (r - m * K) % p - (p if below else 0)
                    if ol.probab_prime(m * K + x):
                        break
                kept.append((m, x))
        m = rng.randrange(1 << 31, 1 << 32)
        while True:  # p times a prime
            m += 1
            x = -(m * K) % p
            if ol.probab_prime((m * K + x) // p):
                break
        dropped += [(m, x), (m, x - p)]
    pairs = kept + dropped
    keep = engine.filter_candidates(fam, np.array([a for a, _ in pairs], dtype=np.uint64),
                                    np.array([b for _, b in pairs], dtype=np.int64), LIMIT)
    assert keep.tolist() == [1] * len(kept) + [0] * len(dropped)
