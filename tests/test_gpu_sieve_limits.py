"""Sieve calls whose limit changes from one to the next on one engine (prime
tables follow the limit, the list staging stays), and both ways that lists come
back: whole, up to 2^18 words of full lists in a batch of up to 4096 m's, or
packed."""
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


# words of full lists: 2 SL count
@pytest.mark.parametrize("SL,count", [(1, 1), (1, 4097), (32, 4096), (32, 4097), (1024, 127), (1024, 128), (1024, 129),
                                      (65535, 2), (65536, 2), (131072, 1), (131073, 1)])
def test_whole_and_packed_lists(engine, SL, count):
    P, D, limit = 101, 210, 1000
    ms = [1 + 2 * i for i in range(count - 1)] + [123456789]
    got = engine.sieve(engine.family(P, D, SL), ms, limit, SL)
    assert len(got) == count
    sv = ol.Sieve(P, D, SL, limit)
    for i in {0, count // 2, count - 2, count - 1} & set(range(count)):
        wp, wn = sv(ms[i])
        assert np.array_equal(got[i][0], wp) and np.array_equal(got[i][1], wn), i
