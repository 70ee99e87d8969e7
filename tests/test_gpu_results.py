"""Results in the dense and the compact layout and of the gapped stage at the
edges of the layout's blocks (4,096 subjects) and of the copies out (what fits
the 64 MiB buffer with one wait and what does not), against the oracle,
bit-exactly."""
import numpy as np
import pytest

import hbseed
import oracle_lib

pytestmark = pytest.mark.gpu

Q = hbseed.random_protein(7980, 60)
SPEC = hbseed.blastp_query(Q, cutoff=20)


@pytest.fixture(scope="module")
def ctx():
    c = hbseed.Context(0)
    yield c
    c.close()


def database(n, length, seed, every):
    """n subjects of `length` residues, every `every`-th (and the last) ending in
    a piece of the query."""
    res = hbseed.random_protein(seed, n * length)
    offs = np.arange(0, (n + 1) * length, length, dtype=np.uint64)
    if every:
        rows = res.reshape(n, length)
        k = min(length, len(Q))
        rows[::every, length - k:] = Q[:k]
        rows[-1, length - k:] = Q[:k]
    return res, offs


def check(ctx, res, offs, gapped=True):
    oq = oracle_lib.OracleQuery.from_spec(SPEC)
    cnt, ref = oq.scan(res, offs, threads=8)
    db = hbseed.Database(ctx, res, offs)
    query = hbseed.Query(ctx, SPEC)
    scan = hbseed.Scan(ctx, db, query)
    stats, hsps = scan.results()
    subjects, hsps2, totals = scan.results_compact()
    assert np.array_equal(hsps.view(np.int32), ref.view(np.int32))
    assert np.array_equal(hsps2.view(np.int32), ref.view(np.int32))
    for i, f in enumerate(("lookup_hits", "extensions", "n_hsp")):
        assert np.array_equal(stats[f], cnt[:, i])
    with_hsps = np.nonzero(cnt[:, 2])[0]
    assert np.array_equal(subjects["oid"], with_hsps)
    assert np.array_equal(subjects["lookup_hits"], cnt[with_hsps, 0])
    assert np.array_equal(subjects["first"], stats["first"][with_hsps])
    assert totals["lookup_hits"] == cnt[:, 0].sum() and totals["extensions"] == cnt[:, 1].sum()
    if gapped:
        gst, g = scan.gapped([30])
        gcnt, gref = oracle_lib.gapped_db(oq, res, offs, ref, [30], threads=8)
        assert np.array_equal(g.view(np.int32), gref.view(np.int32))
        assert np.array_equal(gst["n_hsp"], gcnt[:, 0])
        assert np.array_equal(gst["extensions"], gcnt[:, 1])
    for h in (scan, query, db):
        h.close()
    return len(ref)


@pytest.mark.parametrize("n", [1, 2, 4095, 4096, 4097, 8192, 12289])
@pytest.mark.parametrize("every", [0, 1, 7])
def test_blocks(ctx, n, every):
    found = check(ctx, *database(n, 90, 7981 + n, every))
    assert found or not every


def test_many_records_and_one_large_subject(ctx):
    """More records than the copies before the totals take, and subjects whose
    records the host orders."""
    res, offs = database(30000, 70, 7990, 1)
    big = np.tile(Q, 400)
    res = np.concatenate([big, res, big])
    offs = np.concatenate([[0], offs + np.uint64(len(big)), [len(res)]]).astype(np.uint64)
    assert check(ctx, res, offs, gapped=False) > 30000


def test_results_past_the_pinned_buffer(ctx):
    """Dense results of 70 MB, whose size is no multiple of 64."""
    n = 2900001
    assert (24 * n) % 64 and 24 * n > 64 << 20
    check(ctx, *database(n, 30, 7991, 101))
