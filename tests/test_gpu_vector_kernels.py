"""The one-lane and lane-group kernels against the oracle at every width.  Left to
choose, the engine puts batches below a round of the device, and scans of few
m's, on the matrix cores; here the engine's lanes are fixed, and the parity
tests of batches, graphs, strong Lucas and scans run on it.  Every batch asserts
that no row ran on the matrix cores."""
import random

import numpy as np
import pytest

import oracle_lib as ol
import pgap
import test_gpu_graph as graph
import test_gpu_lucas as lucas
import test_gpu_prp as prp
import test_gpu_scan as scan

pytestmark = pytest.mark.gpu


def fixed(n):
    class Fixed(pgap.Engine):
        def __init__(self, *args, **kw):
            super().__init__(*args, **{"lanes": n, **kw})

        def prp(self, *args, **kw):
            out = super().prp(*args, **kw)
            assert self.last_launch().matrix_tests == 0
            return out

        def prp_device(self, *args, **kw):
            super().prp_device(*args, **kw)
            assert self.last_launch().matrix_tests == 0

    return Fixed


@pytest.fixture(scope="module")
def engines():
    made = {n: fixed(n)(0) for n in (1, 4, 8, 16, 64)}
    yield made
    for e in made.values():
        e.close()


@pytest.fixture
def one_lane(monkeypatch):
    """Engines that a test makes itself."""
    monkeypatch.setattr(pgap, "Engine", fixed(1))


# ---- one lane per number


@pytest.mark.parametrize("digits", [12, 26, 40, 56, 60, 64, 78, 80])
def test_headroom_by_base(engines, digits):
    # numbers of 28 digits - 4 (Fermat), - 8 (bases to 8) and - 14 bits (larger
    # bases), the widest that the lazy bounds admit, on exactly that variant
    rng = random.Random(digits)
    for slack, kind, bases in ((4, pgap.FERMAT2, ()), (8, pgap.SPRP, (3, 5, 7)), (14, pgap.SPRP, (2, 61))):
        bits = 28 * digits - slack
        vals = [rng.getrandbits(bits) | (1 << (bits - 1)) | 1 for _ in range(126)]
        vals += [(1 << bits) - 1, (1 << bits) - 3]
        x = (1 << bits) - 1
        while not ol.probab_prime(x):
            x -= 2
        got = prp.check(engines[1], vals + [x], kind, bases)
        assert got[-1] == 1
        assert (engines[1].last_launch().digits, engines[1].last_launch().lanes_per_number) == (digits, 1)


@pytest.mark.parametrize("bits", [256, 400, 700, 706, 900, 1108, 1120, 1300, 1336, 1400, 1650, 1730, 1750, 1900,
                                  2000, 2129, 2180, 2226])
def test_random_sizes(engines, bits):
    prp.test_random_sizes(engines[1], bits)
    assert engines[1].last_launch().lanes_per_number == 1


def test_families_and_special_values(engines):
    prp.test_special_values_fermat(engines[1])
    prp.test_special_values_sprp(engines[1])
    prp.test_config_families(engines[1])
    prp.test_large_family_and_sprp(engines[1])


@pytest.mark.parametrize("kind,bases,bits", [(pgap.FERMAT2, (), 1108), (pgap.SPRP, (3, 5), 1108),
                                             (pgap.SPRP, (2, 3, 5), 2128)])
def test_graph_replay(one_lane, kind, bases, bits):
    graph.test_replay_matches_eager(kind, bases, bits)


# the engine's own choice: a round of 65536 rows on one lane each, 37 more on the
# matrix cores; later bases divide their survivors on the device
@pytest.mark.parametrize("bits", [300, 705, 1108, 1560, 2128])
@pytest.mark.parametrize("kind,bases", [(pgap.FERMAT2, ()), (pgap.SPRP, (2, 3)), (pgap.BPSW, ())])
def test_full_round_of_the_default_engine(engine, bits, kind, bases):
    rng = random.Random(bits)
    vals = [rng.getrandbits(bits) | (1 << (bits - 1)) | 1 for _ in range(500)]
    for q in (521, 607, 1279, 127, 89):
        vals.append((1 << q) - 1 if q <= bits else (1 << 61) - 1)
    vals += [2047, 1, 2, 0]  # 509 rows
    arr = pgap.to_limbs(vals, (bits + 31) // 32)
    rows = np.resize(arr, (65536 + 37, arr.shape[1]))
    got = engine.prp(rows, kind, bases)
    assert np.array_equal(got, np.resize(ol.verdicts(arr, kind, bases), len(rows)))
    assert engine.last_launch().matrix_tests == 37


# mixed buckets of one lane per number, up to their last bit
@pytest.mark.parametrize("digits,rows", [(12, 4000), (26, 12000), (40, 17000), (56, 31000), (78, 46000)])
@pytest.mark.parametrize("slack,kind,bases", [(4, pgap.FERMAT2, ()), (8, pgap.SPRP, (3,)), (14, pgap.SPRP, (61,))])
def test_mixed_bucket_edges(engine, digits, rows, slack, kind, bases):
    bits = 28 * digits - slack
    rng = random.Random(bits)
    vals = [rng.getrandbits(bits) | (1 << (bits - 1)) | 1 for _ in range(61)] + [(1 << bits) - 1, 2047]
    x = (1 << bits) - 1
    while not ol.probab_prime(x):
        x -= 2
    vals.append(x)
    arr = pgap.to_limbs(vals, (bits + 31) // 32)
    i = np.arange(rows) % len(vals)
    got = engine.prp_mixed_packed(arr.reshape(-1), i * arr.shape[1], np.full(rows, arr.shape[1]), kind, bases)
    assert np.array_equal(got, ol.verdicts(arr, kind, bases)[i])
    assert engine.last_launch().matrix_tests == 0


# ---- lane groups


@pytest.mark.parametrize("bits", [2300, 2490, 2600, 2680, 3000, 3320, 3352])
def test_quad_widths(engines, bits):
    rng = random.Random(bits)
    vals = [rng.getrandbits(bits) | (1 << (bits - 1)) | 1 for _ in range(60)] + [(1 << 2281) - 1, (1 << 2203) - 1]
    for kind, bases in ((pgap.FERMAT2, ()), (pgap.SPRP, (2, 3))):
        got = prp.check(engines[4], vals, kind, bases)
        assert got[-2:].all() and engines[4].last_launch().lanes_per_number == 4


@pytest.mark.parametrize("lanes", [8, 16, 64])
def test_lucas_families(engines, lanes):
    e = engines[lanes]
    vals = list(range(0, 3000)) + lucas.STRONG_LUCAS_PSP + lucas.SPSP_235
    lucas.check(e, vals, pgap.LUCAS)
    lucas.check(e, vals, pgap.BPSW)
    lucas.test_pseudoprimes_squares_and_special_forms(e)
    for bits in (30, 200, 894, 1108, 1800, 2186, 2236, 3576, 4470):
        lucas.test_random_sizes(e, bits)


# ---- scans on one-lane rounds and lane-group Lucas tests


@pytest.mark.parametrize("confirm", [pgap.CONFIRM_NONE, pgap.CONFIRM_SPRP2, pgap.CONFIRM_BPSW])
def test_scan_confirmations(one_lane, confirm):
    scan.test_confirmation_rejects_fermat_pseudoprimes(confirm)
    if confirm != pgap.CONFIRM_SPRP2:
        scan.test_width_grows_past_a_power_of_two(confirm)


def test_scan_rows(one_lane, unknowns_907):
    scan.test_scan_rows_907_match_oracle(unknowns_907)
    scan.test_scan_depth_and_confirmation_do_not_change_rows(unknowns_907, 3, pgap.CONFIRM_SPRP2)
    scan.test_bpsw_confirmation_rejects_strong_pseudoprimes()
    scan.test_small_centres_fall_back_to_small_primes()
    scan.test_side_skip_follows_gap_test_gpu_rule(unknowns_907, 6.0)
    scan.test_fallback_beyond_sieve_length()
    scan.test_scan_2100_bit_family_small()
    scan.test_one_sided_requests_return_their_half(unknowns_907)
