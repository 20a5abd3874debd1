"""Which scans run their rounds on the matrix cores, seen in the tests that a
scan issues: a matrix round holds some 2048 numbers, a one-lane round 65536."""
import numpy as np
import pytest

import oracle_lib as ol
import pgap

pytestmark = pytest.mark.gpu


def scan(P, d, SL, m, xs, confirm, **options):
    """Rows and tests issued of one m whose sides may each issue their whole list in a round."""
    with pgap.Engine(0, **options) as e:
        fam = e.family(P, d, SL)
        e.scan_config(4096, confirm)
        assert e.scan_submit(fam, m, xs, xs) == pgap.PGAP_OK
        (r,) = e.scan_poll(wait=True)
        return (r.prev_p, r.next_p, r.p_tests, r.n_tests), e.scan_stats()["tests_issued"]


# m * P#/d is even or odd; every odd offset that keeps N odd is a candidate
def offsets(P, d, m, SL):
    return np.arange(1 + (m * ol.K(P, d)) % 2, SL, 2, dtype=np.int32)


@pytest.mark.parametrize("confirm", [pgap.CONFIRM_BPSW, pgap.CONFIRM_NONE])
def test_an_occupancy_cap_keeps_the_matrix_rounds(confirm):
    P, d, SL, m = 503, 210, 8000, 101
    xs = offsets(P, d, m, SL)
    row, issued = scan(P, d, SL, m, xs, confirm)
    capped_row, capped = scan(P, d, SL, m, xs, confirm, waves_per_simd=1)
    lane_row, lane = scan(P, d, SL, m, xs, confirm, lanes=1)
    want = ol.test_interval(P, d, m, SL, xs, xs, kind=0)
    assert row == capped_row == lane_row == (want["prev_p"], want["next_p"], want["p_tests"], want["n_tests"])
    assert issued < 4000 and lane >= 2 * len(xs) - 200
    assert abs(capped - issued) < 1000  # the same rounds; a Lucas test may end in another one


@pytest.mark.parametrize("P,confirm,matrix", [(101, pgap.CONFIRM_BPSW, True), (101, pgap.CONFIRM_SPRP2, False),
                                              (101, pgap.CONFIRM_NONE, False), (251, pgap.CONFIRM_SPRP2, True),
                                              (251, pgap.CONFIRM_NONE, True)])
def test_narrow_numbers_without_lucas_tests_stay_on_one_lane(P, confirm, matrix):
    d, SL, m = 210, 8000, 101
    xs = offsets(P, d, m, SL)
    row, issued = scan(P, d, SL, m, xs, confirm)
    want = ol.test_interval(P, d, m, SL, xs, xs, kind=0)
    assert row == (want["prev_p"], want["next_p"], want["p_tests"], want["n_tests"])
    assert issued < 4000 if matrix else issued >= 2 * len(xs) - 200
