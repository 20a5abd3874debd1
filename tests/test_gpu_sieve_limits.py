"""Sieve calls whose limit changes from one to the next on one engine: prime
tables follow the limit, the list staging stays."""
import numpy as np
import pytest

import oracle_lib as ol
import pgap

pytestmark = pytest.mark.gpu


def test_limits_in_turn():
    fams = [(503, 210, 4000, [1, 11, 13]), (1511, 2190, 9000, [1, 7])]
    limits = [10_000, 300_000, 10_000, 2_000_000, 1000]
    with pgap.Engine(0) as e:
        for limit in limits:
            for P, D, SL, ms in fams:
                sv = ol.Sieve(P, D, SL, limit)
                for m, (p, n) in zip(ms, e.sieve(e.family(P, D, SL), ms, limit, SL)):
                    wp, wn = sv(m)
                    assert np.array_equal(p, wp) and np.array_equal(n, wn), (P, limit, m)
