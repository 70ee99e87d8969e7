"""Scans whose diagonals are split into classes: query lengths on both sides
of each change of the number of classes, plain and batched (beside queries of
one class), windows of 4 and 255, subjects shorter than a word, of one tile
and longer than the staging ring, against the oracle, bit-exactly."""
import numpy as np
import pytest

import hbseed
import oracle_lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    c = hbseed.Context(0)
    pq = hbseed.random_protein(9901, 1500)
    res, offs = hbseed.make_db(9900, 1200, median=120.0, sigma=1.3, lo=1, hi=9000,
                               plant_query=pq, plant_frac=0.2)
    db = hbseed.Database(c, res, offs)
    yield c, db, pq, res, offs
    db.close()
    c.close()


def spec_of(n, pq):
    q = hbseed.random_protein(9910 + n, n)
    k = min(n, len(pq)) // 2
    q[n - k:] = pq[:k]   # homologs on the last diagonals too
    return hbseed.blastp_query(q)


def check(stats, hsps, cnt, ref):
    assert len(ref) > 0
    assert np.array_equal(hsps.view(np.int32), ref.view(np.int32))
    assert np.array_equal(stats["lookup_hits"], cnt[:, 0])
    assert np.array_equal(stats["extensions"], cnt[:, 1])
    assert np.array_equal(stats["n_hsp"], cnt[:, 2])


@pytest.mark.parametrize("n", [1520, 1600, 3111, 3300, 5999, 6300, 11003, 13000, 19009, 23001, 31001])
def test_plain(setup, n):
    c, db, pq, res, offs = setup
    spec = spec_of(n, pq)
    cnt, ref = oracle_lib.OracleQuery.from_spec(spec).scan(res, offs, threads=8)
    q = hbseed.Query(c, spec)
    for mode in (hbseed.STATE_AUTO, hbseed.STATE_GLOBAL):
        q.set_state_mode(mode)
        s = hbseed.Scan(c, db, q)
        check(*s.results(), cnt, ref)
        s.close()
    q.close()


@pytest.mark.parametrize("window", [4, 255])
@pytest.mark.parametrize("n", [2501, 9000])
def test_windows(setup, n, window):
    c, db, pq, res, offs = setup
    spec = spec_of(n, pq)
    cnt, ref = oracle_lib.OracleQuery.from_spec(spec, window=window).scan(res, offs, threads=8)
    q = hbseed.Query(c, spec, window=window)
    s = hbseed.Scan(c, db, q)
    check(*s.results(), cnt, ref)
    s.close()
    q.close()


def test_table_of_classes(setup):
    c, _, pq, _, _ = setup
    spec = spec_of(6300, pq)
    q = hbseed.Query(c, spec)
    start, ent = q.lut()
    q.close()
    ostart, oent = oracle_lib.OracleQuery.from_spec(spec).lut_arrays()
    assert np.array_equal(start, ostart) and np.array_equal(ent, oent)


def test_batched_beside_short(setup):
    c, db, pq, res, offs = setup
    specs = [spec_of(n, pq) for n in (90, 700, 1400, 1700, 3300, 7001, 14000, 25000)]
    b = hbseed.Batch(c, db, group_residues=768)
    ids = [b.add(s) for s in specs]
    b.run()
    for i, s in zip(ids, specs):
        _, ref = oracle_lib.OracleQuery.from_spec(s).scan(res, offs, threads=8)
        assert np.array_equal(b.results(i).view(np.int32), ref.view(np.int32))
    b.close()
