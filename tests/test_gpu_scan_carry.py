"""Carries and borrows across the words of a scan's N = centre -+ x: centres of
zeros or ones in every low word, against the oracle's rows."""
import numpy as np
import pytest

import oracle_lib as ol
import pgap

pytestmark = pytest.mark.gpu

# (P, d, m, centre m * P#/d)
CENTRES = [(11, 1155, 1 << 31, 1 << 32),
           (11, 1155, 1 << 62, 1 << 63),
           (11, 1155, (1 << 31) - 1, (1 << 32) - 2),
           (5, 2, 0x11111111, (1 << 32) - 1),
           (5, 2, 0x1111111111111111, (1 << 64) - 1)]


@pytest.mark.parametrize("P,d,m,centre", CENTRES)
def test_carry_chain(P, d, m, centre):
    assert m * ol.K(P, d) == centre
    SL = 200
    xs = list(range(1 + centre % 2, SL, 2))  # every odd N
    want = ol.test_interval(P, d, m, SL, xs, xs, kind=0)
    with pgap.Engine(0) as e:
        fam = e.family(P, d, SL)
        e.scan_submit(fam, m, np.array(xs, np.int32), np.array(xs, np.int32), tag=m)
        (r,) = e.scan_poll(wait=True)
    assert (r.m, r.prev_p, r.next_p, r.p_tests, r.n_tests) == \
        (m, want["prev_p"], want["next_p"], want["p_tests"], want["n_tests"])
