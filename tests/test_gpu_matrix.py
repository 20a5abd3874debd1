"""Matrix-core variants (one number per wavefront, csrc/mont_mf.h) against the
oracle: widths at the edges of every container, and batches cut between whole
rounds of the one-lane variant and a remainder on the matrix cores."""
import random

import numpy as np
import pytest

import oracle_lib as ol
import pgap

pytestmark = pytest.mark.gpu

MERSENNE = [521, 607, 1279, 2203, 2281, 3217, 4253, 4423]


def check(engine, vals, kind, bases=(), limbs=None):
    arr = pgap.to_limbs(vals, limbs or max(pgap.limbs_needed(v) for v in vals))
    got = engine.prp(arr, kind, bases)
    want = ol.verdicts(arr, kind, bases)
    bad = np.nonzero(got != want)[0]
    assert len(bad) == 0, [(hex(vals[i]), int(got[i]), int(want[i])) for i in bad[:5]]
    return got


# containers of 16 k - 1 words (15, 31, 63, ...) or 16 k + 1 (49, 145) take 32
# words - 16 bits; 4466 is the widest that every base takes
@pytest.mark.parametrize("top", [464, 976, 1488, 1552, 2000, 2512, 3024, 3536, 4048, 4466])
def test_container_edges(engine, top):
    rng = random.Random(top)
    vals = [(1 << top) - 1, (1 << top) - 3, (1 << (top - 1)) + 1, (1 << top) - (1 << (top // 2)) - 1]
    vals += [rng.getrandbits(b) | (1 << (b - 1)) | 1 for b in (top, top, top - 1, top - 15, top - 16, top - 31, 257)]
    # every word of the quotient at the ends of the balanced range
    vals += [int.from_bytes(bytes([c]) * (top // 8 - 1), "little") | 1 for c in (0x7F, 0x80, 0x81, 0xFF)]
    vals += [0, 1, 2, 3, 5, 9, 341, 561, 2047, 3277, 25326001, 3215031751, (1 << 61) - 1, (1 << 89) - 1]
    vals += [(1 << p) - 1 for p in MERSENNE if p <= top]
    vals += [3 * ((1 << p) - 1) for p in MERSENNE if p + 2 <= top]
    limbs = (top + 31) // 32
    for kind, bases in ((pgap.FERMAT2, ()), (pgap.SPRP, (2,)), (pgap.SPRP, (3, 5)), (pgap.SPRP, (2, 61))):
        got = check(engine, vals, kind, bases, limbs)
        assert engine.last_launch().matrix_tests == len(vals)
        primes = [i for i, v in enumerate(vals) if v in {(1 << p) - 1 for p in MERSENNE}]
        assert got[primes].all()


@pytest.mark.parametrize("kind,bases", [(pgap.FERMAT2, ()), (pgap.SPRP, (3, 7))])
def test_remainder_of_a_round(engine, kind, bases):
    # 65536 rows are a round of one-lane wavefronts: one row, and the rows of
    # a nearly full second round, beyond it
    rng = random.Random(len(bases))
    bits = 300
    vals = [rng.getrandbits(bits) | (1 << (bits - 1)) | 1 for _ in range(4096)]
    vals[4095] = vals[0] = vals[17] = (1 << 127) - 1
    vals[1], vals[2], vals[3] = 2047, 4, 1
    arr = pgap.to_limbs(vals, (bits + 31) // 32)
    want = ol.verdicts(arr, kind, bases)
    for count in (65536, 65537, 65536 + 1000, 2 * 65536 - 1):
        rows = np.resize(arr, (count, arr.shape[1]))
        got = engine.prp(rows, kind, bases)
        assert np.array_equal(got, np.resize(want, count)), count
        assert engine.last_launch().matrix_tests == (count - 65536 if count - 65536 <= 1000 else 0)


@pytest.mark.parametrize("top", [464, 976, 1488, 1552, 2000, 2512, 3024, 3536, 4048, 4472])
def test_strong_lucas_edges(engine, top):
    # the Lucas chain's set-up (parameter search, 1 / Q, N = 2^b - 1) and its
    # width bounds, against the oracle and the lane variant's bound of 4472
    rng = random.Random(100 + top)
    vals = list(range(0, 130)) + [5459, 5777, 10877, 16109, 18971, 1093 ** 2, 3511 ** 2, (1 << 61) - 1]
    vals += [(1 << top) - 1, (1 << top) - 3, (1 << (top - 1)) + 1, (rng.getrandbits(top // 2) | 1) ** 2]
    vals += [rng.getrandbits(b) | (1 << (b - 1)) | 1 for b in (top, top, top - 15, top - 31)]
    vals += [(1 << p) - 1 for p in MERSENNE if p <= top] + [3 * ((1 << p) - 1) for p in MERSENNE if p + 2 <= top]
    # primes whose parameter D is large: N = 1 mod 4 and mod the odd primes below 30, 44 and 60
    for below in (30, 44, 60):
        M = 4
        for p in range(3, below, 2):
            if all(p % q for q in range(3, p, 2)):
                M *= p
        v = 1 + M * rng.getrandbits(min(top, 700) - M.bit_length())
        while not ol.probab_prime(v):
            v += M
        vals.append(v)
    limbs = (top + 31) // 32
    got = check(engine, vals, pgap.LUCAS, (), limbs)
    assert got[-3:].all() and engine.last_launch().matrix_tests == len(vals)
    check(engine, vals, pgap.BPSW, (), limbs)


@pytest.mark.parametrize("kind,bases", [(pgap.FERMAT2, ()), (pgap.SPRP, (2, 61))])
def test_mixed_batch_on_both_kernels(engine, kind, bases):
    # a one-lane bucket with more rows than the matrix cores take, beside
    # buckets of a few rows and one number at every container's width
    rng = random.Random(7)
    vals = [rng.getrandbits(300) | (1 << 299) | 1 for _ in range(5000)]
    vals += [rng.getrandbits(b) | (1 << (b - 1)) | 1 for b in (700, 720, 1100, 2100, 2180, 2250, 4400)]
    vals += [rng.getrandbits(32 * (16 * k - 1) - 16) | 1 for k in range(1, 9)] + [rng.getrandbits(b) | 1 for b in (1489, 1552, 1553)]
    vals += [(1 << p) - 1 for p in MERSENNE] + [3 * ((1 << p) - 1) for p in MERSENNE] + [0, 1, 2, 3, 5, 2047, 341]
    rng.shuffle(vals)
    got = engine.prp_mixed([pgap.to_limbs([v], pgap.limbs_needed(v))[0] for v in vals], kind, bases)
    if kind == pgap.FERMAT2:
        assert 0 < engine.last_launch().matrix_tests < 100
    want = ol.verdicts(pgap.to_limbs(vals, 140), kind, bases)
    bad = np.nonzero(got != want)[0]
    assert len(bad) == 0, [(hex(vals[i])[:40], vals[i].bit_length(), int(got[i]), int(want[i])) for i in bad[:5]]
