"""The trial-division screen of pairs outside the fixed-point range (m >= 2^32 or
|x| >= 2^31) through its three stages and the compaction between them."""
import math
import random

import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu


def with_factor(top, limit):
    """bad[n]: some prime <= limit divides n, for n below top."""
    bad = np.zeros(top, dtype=bool)
    for p in range(2, limit + 1):
        if p * p > limit or not bad[p]:
            if all(p % q for q in range(2, math.isqrt(p) + 1)):
                bad[::p] = True
    return bad


# 524288 candidates are one pass of the compaction's grid
@pytest.mark.parametrize("count", [1, 1023, 1025, 600_001])
def test_wide_and_fixed_forms_agree(engine, count):
    # N = 2 m + x for 11#/1155: (m + 2^32, x - 2^33) is the same N
    limit, top = 100_003, 4_000_000
    fam = engine.family(11, 1155, 0)
    rng = np.random.default_rng(count)
    first, bad = with_factor(top, 1023), with_factor(top, limit)
    N = rng.choice(np.nonzero(~first)[0], size=count).astype(np.int64)  # all reach the second stage
    N[::17] = rng.integers(0, top, size=len(N[::17]))
    m = rng.integers(1, 1_000_000, size=count)
    x = N - 2 * m
    kinds = rng.integers(0, 4, size=count)
    kinds[: count // 100] = 0
    shift = np.choose(kinds, [0, 1 << 32, 1 << 30, 1 << 40])  # fixed; m and x wide; x wide; both
    keep = engine.filter_candidates(fam, (m + shift).astype(np.uint64), x - 2 * shift, limit)
    assert np.array_equal(keep != 0, ~bad[N])


@pytest.mark.parametrize("limit", [1009, 1031, 32771, 40009])
def test_wide_matches_big_integers(engine, limit):
    P, D = 101, 210
    K, fam = ol.K(P, D), engine.family(P, D, 0)
    prod = math.prod(p for p in range(2, limit + 1) if all(p % q for q in range(2, math.isqrt(p) + 1)))
    low = math.prod(p for p in range(2, 200) if all(p % q for q in range(2, math.isqrt(p) + 1)))
    rng = random.Random(limit)
    pairs = []
    while len(pairs) < 3000:
        m = rng.choice([rng.randrange(1 << 32, 1 << 64), rng.randrange(1, 1 << 32), (1 << 64) - 1 - len(pairs)])
        x = rng.choice([rng.randrange(-(1 << 31), 1 << 31), rng.randrange(-(1 << 63), 1 << 63)])
        if len(pairs) % 3 == 0 or math.gcd(abs(m * K + x), low) == 1:
            pairs.append((m, x))
    keep = engine.filter_candidates(fam, np.array([p[0] for p in pairs], dtype=np.uint64),
                                    np.array([p[1] for p in pairs], dtype=np.int64), limit)
    assert keep.tolist() == [int(math.gcd(abs(a * K + b), prod) == 1) for a, b in pairs]
