"""Work distribution of the scans: databases around the number of tile
queues and of wavefronts (plain form), and batches whose groups are fewer,
as many and more than the streams that share them (batched form), against
the oracle, bit-exactly."""
import numpy as np
import pytest

import hbseed
import oracle_lib

from test_gpu_parity import compare

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hbseed.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 4095, 4097, 9000])
def test_plain_database_sizes(ctx, n):
    q = hbseed.random_protein(9100 + n, 220)
    # lengths from 1 up: the shortest tiles hold 64 subjects, the longest one
    res, offs = hbseed.make_db(9200 + n, n, median=60.0, sigma=1.4, lo=1, hi=9000,
                               plant_query=q, plant_frac=0.2)
    compare(ctx, hbseed.blastp_query(q), res, offs)


@pytest.mark.parametrize("n_queries", [1, 7, 8, 9, 70])
@pytest.mark.parametrize("n", [3, 2500])
def test_batched_group_counts(ctx, n_queries, n):
    queries = [hbseed.random_protein(9300 + i, 40 + 11 * (i % 30)) for i in range(n_queries)]
    res, offs = hbseed.make_db(9400 + n, n, median=90.0, sigma=1.0, lo=1, hi=6000,
                               plant_query=queries[0], plant_frac=0.2)
    db = hbseed.Database(ctx, res, offs)
    batch = hbseed.Batch(ctx, db, group_residues=64)   # every query its own group
    ids = [batch.add(hbseed.blastp_query(q)) for q in queries]
    batch.run()
    assert batch.info()["n_groups"] == n_queries
    for _ in range(2):   # the first pass and a replay
        for i, q in zip(ids, queries):
            _, ref = oracle_lib.OracleQuery.from_spec(hbseed.blastp_query(q)).scan(res, offs)
            assert np.array_equal(batch.results(i).view(np.int32), ref.view(np.int32))
        batch.run()
    batch.close()
    db.close()
