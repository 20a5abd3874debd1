"""Which buckets of a mixed call run one lane per number and which on the matrix
cores: the whole call decides, not each bucket against a round of its own."""
import random

import numpy as np
import pytest

import oracle_lib as ol
import pgap

pytestmark = pytest.mark.gpu


# (bits, rows), and whether the width runs on the matrix cores
@pytest.mark.parametrize("spec", [
    [(1110, 20000, False)], [(1110, 8000, True)], [(1560, 32000, False)], [(1560, 20000, True)],
    [(330, 3300, False), (720, 11000, False), (1110, 20000, False)],
    [(330, 3300, False), (720, 11000, False), (1110, 20000, False), (1560, 32000, False), (2128, 39000, False)],
    [(330, 800, True), (720, 2700, True), (1110, 5000, True), (1560, 8000, True), (2128, 9500, True)],
    [(2128, 60000, False), (1110, 500, False), (330, 5, False), (4247, 64, True)],
    [(720, 131072, False), (2128, 29, True), (2180, 3, True)],
    [(200, 100, False), (2128, 29, True)], [(200, 100, False)], [(2, 64, True), (300, 65, True)],  # one bucket, its widest row decides
])
def test_split(engine, spec):
    rng = random.Random(len(spec))
    words, offset, limbs, want, matrix = [], [], [], [], 0
    at = 0
    for bits, rows, mx in spec:
        vals = [rng.getrandbits(bits) | (1 << (bits - 1)) | 1 for _ in range(29)]
        x = vals[0]
        while not ol.probab_prime(x) or x.bit_length() != bits:
            x = x + 2 if x.bit_length() == bits else 1 << (bits - 1) | 1
        vals.append(x)
        L = (bits + 31) // 32
        arr = pgap.to_limbs(vals, L)
        words.append(arr.reshape(-1))
        i = np.arange(rows) % len(vals)
        offset.append(at + i * L)
        limbs.append(np.full(rows, L))
        want.append(ol.verdicts(arr)[i])
        at += arr.size
        matrix += rows if mx else 0
    perm = np.random.default_rng(1).permutation(sum(len(o) for o in offset))
    got = engine.prp_mixed_packed(np.concatenate(words), np.concatenate(offset)[perm], np.concatenate(limbs)[perm])
    assert np.array_equal(got, np.concatenate(want)[perm])
    assert engine.last_launch().matrix_tests == matrix
