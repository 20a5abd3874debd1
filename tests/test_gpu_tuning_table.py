"""Which kernel a loaded tuning table puts a batch on: a lane group of the table
runs every row unless its entry has the matrix cores faster; one lane per number
runs whole rounds and leaves the remainder to the matrix cores."""
import random

import numpy as np
import pytest

import oracle_lib as ol
import pgap

pytestmark = pytest.mark.gpu

BASES = {pgap.FERMAT2: (), pgap.SPRP: (2, 3), pgap.LUCAS: ()}


def tuned(tmp_path, *lines):
    path = tmp_path / "pgap.tune"
    path.write_text("# comment\n" + "\n".join(lines) + "\n")
    return pgap.Engine(0, tuning_path=str(path))


def rows(bits, count, seed=1):
    rng = random.Random(seed * bits)
    vals = [rng.getrandbits(bits) | (1 << (bits - 1)) | 1 for _ in range(count - 1)]
    vals.append(next(p for p in ((1 << q) - 1 for q in (4423, 4253, 3217, 2203, 1279, 607, 127, 61)) if p.bit_length() <= bits))
    return pgap.to_limbs(vals, (bits + 31) // 32)


def check(e, arr, kind, matrix):
    got = e.prp(arr, kind, BASES[kind])
    assert np.array_equal(got, ol.verdicts(arr, kind, BASES[kind])) and got[-1] == 1
    assert e.last_launch().matrix_tests == (len(arr) if matrix else 0)


# (digits, lanes) of 28 bits; the last field is the matrix cores' rate
@pytest.mark.parametrize("bits", [2128, 4247])
@pytest.mark.parametrize("matrix", ["", " 0.0", " 999.0", " 1001.0"])
def test_lane_group_entries(tmp_path, bits, matrix):
    with tuned(tmp_path, f"0 4300 28 160 8 0 1000.0{matrix}", f"1 4300 28 160 16 0 1000.0{matrix}",
               f"2 4300 28 160 16 0 1000.0{matrix}") as e:
        faster = matrix.strip() == "1001.0"
        arr = rows(bits, 150)
        for kind, lanes in ((pgap.FERMAT2, 8), (pgap.SPRP, 16), (pgap.LUCAS, 16)):
            check(e, arr, kind, faster)
            if not faster or bits > 2232 or kind == pgap.LUCAS:
                assert e.last_launch().lanes_per_number == lanes
        got = e.prp(arr, pgap.BPSW)
        assert np.array_equal(got, ol.verdicts(arr, pgap.BPSW))


def test_one_lane_entry_keeps_the_remainder_rule(tmp_path):
    with tuned(tmp_path, "0 300 28 12 1 0 1000.0") as e:
        arr = rows(300, 200)
        check(e, arr, pgap.FERMAT2, True)
        full = np.resize(arr, (65536 + 200, arr.shape[1]))
        assert np.array_equal(e.prp(full), np.resize(ol.verdicts(arr), len(full)))
        assert e.last_launch().matrix_tests == 200
    with tuned(tmp_path, "0 300 28 12 1 0 1000.0 1001.0") as e:  # the matrix cores throughout
        assert np.array_equal(e.prp(full), np.resize(ol.verdicts(arr), len(full)))
        assert e.last_launch().matrix_tests == len(full)


def test_wide_matrix_entry_leaves_narrow_numbers_one_lane(tmp_path):
    with tuned(tmp_path, "0 4300 28 152 4 0 1000.0 2000.0") as e:
        arr = rows(300, 64)
        full = np.resize(arr, (65536, arr.shape[1]))
        assert np.array_equal(e.prp(full), np.resize(ol.verdicts(arr), len(full)))
        assert e.last_launch().matrix_tests == 0 and e.last_launch().lanes_per_number == 1
        check(e, rows(4247, 40), pgap.FERMAT2, True)


def test_autotune_times_the_matrix_cores(tmp_path):
    with pgap.Engine(0) as e:
        table = e.autotune([200, 2300])
        for r in table:
            assert (r["matrix_tests_per_s"] > 0) == (r["test"] == pgap.LUCAS or r["bits"] >= 256), r
            arr = rows(r["bits"], 100)
            e.prp(arr, r["test"], BASES[r["test"]])
            group_wins = r["lanes"] != 1 and r["tests_per_s"] >= r["matrix_tests_per_s"]
            narrow = r["test"] != pgap.LUCAS and r["bits"] < 256
            assert e.last_launch().matrix_tests == (0 if group_wins or narrow else 100), r


def test_scan_with_a_lane_group_table(tmp_path):
    # 1200 scanning sides: rounds above and below the matrix cores' threshold
    P, d, SL, limit = 101, 210, 1500, 100_000
    ms = [m for m in range(1_000_000, 1_010_000) if all(m % q for q in (2, 3, 5, 7))][:600]
    found = []
    with tuned(tmp_path, "0 400 28 80 8 0 1000.0", "1 400 28 80 8 0 1000.0", "2 400 28 80 8 0 1000.0") as t, \
            pgap.Engine(0) as plain:
        for e in (t, plain):
            fam = e.family(P, d, SL)
            lists = e.sieve(fam, ms, limit, SL)
            for m, (p, n) in zip(ms, lists):
                assert e.scan_submit(fam, m, p, n, tag=m) == pgap.PGAP_OK
            got = []
            while len(got) < len(ms):
                got += e.scan_poll(wait=True)
            found.append(sorted((r.m, r.prev_p, r.next_p, r.p_tests, r.n_tests) for r in got))
    assert found[0] == found[1]
    for m, pp, np_, pt, nt in found[0][::97]:
        p, n = lists[ms.index(m)]
        want = ol.test_interval(P, d, m, SL, p, n, kind=0)
        assert (pp, np_, pt, nt) == (want["prev_p"], want["next_p"], want["p_tests"], want["n_tests"])
