"""The device order of a batched pass's records: record counts around the
sort's steps (64, 1,024 and 4,096 keys) up to more than fit the page-locked
results, one query and many, several contexts, queries without records,
against the oracle, bit-exactly."""
import numpy as np
import pytest

import hbseed
import oracle_lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hbseed.Context(0)
    yield c
    c.close()


def run(ctx, specs, res, offs, group=512):
    db = hbseed.Database(ctx, res, offs)
    b = hbseed.Batch(ctx, db, group_residues=group)
    ids = [b.add(s) for s in specs]
    total = 0
    for _ in range(2):
        b.run()
        total = 0
        for i, s in zip(ids, specs):
            _, ref = oracle_lib.OracleQuery.from_spec(s).scan(res, offs, threads=8)
            assert np.array_equal(b.results(i).view(np.int32), ref.view(np.int32))
            total += len(ref)
        assert b.info()["hsps"] == total
    b.close()
    db.close()
    return total


# cutoff 1: every extension is a record (0, 9, 74, 1,002, 1,062, 4,406, 4,983
# and 102,214 of them)
@pytest.mark.parametrize("n", [1, 3, 14, 200, 210, 900, 1000, 20000])
def test_one_query(ctx, n):
    q = hbseed.random_protein(9950, 200)
    res, offs = hbseed.make_db(9951, n, median=250.0, lo=1, plant_query=q, plant_frac=0.3)
    run(ctx, [hbseed.blastp_query(q, cutoff=1)], res, offs)


def test_many_queries(ctx):
    res, offs = hbseed.make_db(9960, 500, plant_query=hbseed.random_protein(9961, 300),
                               plant_frac=0.2)
    specs = [hbseed.blastp_query(hbseed.random_protein(9962 + i, 20 + i % 90), cutoff=1)
             for i in range(300)]
    specs[7] = hbseed.blastp_query(np.array([1, 2], np.uint8))   # no word, no record
    specs[299] = hbseed.blastp_query(np.array([3], np.uint8))
    specs[40] = hbseed.blastx_query(hbseed.blastx_nt(9963, 900, hbseed.random_protein(9964, 90),
                                                     hbseed.random_protein(9965, 90)), cutoff=1)
    run(ctx, specs, res, offs)


def test_more_than_the_page_locked_results(ctx):
    q = hbseed.random_protein(9970, 900)
    res, offs = hbseed.make_db(9971, 9000, plant_query=q, plant_frac=0.2)
    specs = [hbseed.blastp_query(hbseed.random_protein(9972, 500), cutoff=1),
             hbseed.blastp_query(q, cutoff=1)]
    assert run(ctx, specs, res, offs) * 32 > 12 << 20
