"""A served batch whose budget has no room for ordering its records on the
device orders them on the host: the results equal the oracle's, bit-exactly,
and the budget holds."""
import numpy as np
import pytest

import hbseed
import oracle_lib

pytestmark = pytest.mark.gpu

TABLES = 32768 * 8 + 1024 * 4 + 1024 * 4 + 8192   # of one group, and what else it holds


@pytest.mark.parametrize("room", [1000, 64 << 20])
def test_order_within_the_budget(room):
    q = hbseed.random_protein(9300, 400)
    res, offs = hbseed.make_db(9301, 6000, plant_query=q, plant_frac=0.2)
    # two queries that share subjects, and one that has few of its own
    specs = [hbseed.blastp_query(q), hbseed.blastp_query(hbseed.homolog(9302, q, 0.8, 1)[:400]),
             hbseed.blastp_query(q[::-1].copy())]
    refs = [oracle_lib.OracleQuery.from_spec(s).scan(res, offs, threads=8)[1] for s in specs]
    cells = sum(len(s.seq) for s in specs) * float(len(res))
    per_cell = 1.5 * sum(len(r) for r in refs) / cells
    est = sum(32 * (int(per_cell * len(s.seq) * float(len(res))) + 256) + TABLES + 256 * len(s.seq)
              for s in specs)
    assert 56 * sum(len(r) for r in refs) > 1000
    with hbseed.Context(0) as ctx:
        db = hbseed.Database(ctx, res, offs)
        with hbseed.Server(ctx, db, mem_budget=est + room, max_inflight=1, hsp_per_cell=per_cell,
                           max_batch_queries=len(specs), linger_us=2_000_000) as srv:
            tickets = [srv.submit(s) for s in specs]
            for t, ref in zip(tickets, refs):
                assert srv.wait(t, 60000)
                got = srv.results(t)
                assert len(ref) > 0
                assert np.array_equal(got.view(np.int32), ref.view(np.int32))
            st = srv.stats()
        db.close()
    assert st["batches"] == 1
    assert st["peak_bytes"] <= est + room
    assert (st["peak_bytes"] > est) == (room > 1000)
