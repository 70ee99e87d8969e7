"""The dense layout's records have no bytes that nothing wrote: the four of
hb_subject_stats between n_hsp and first are 0 whatever the result buffers
held before."""
import numpy as np
import pytest

import hbseed

pytestmark = pytest.mark.gpu


def test_padding_is_zero():
    q = hbseed.random_protein(9400, 300)
    spec = hbseed.blastp_query(q)
    with hbseed.Context(0) as ctx:
        # loads and searches of sizes that hand the same buffers round
        for n in (2000, 3000, 1500, 2500, 5000, 2000):
            res, offs = hbseed.make_db(9401 + n, n, plant_query=q, plant_frac=0.2)
            db = hbseed.Database(ctx, res, offs)
            for _ in range(3):
                stats, _ = hbseed.search(ctx, db, spec)
                raw = np.ascontiguousarray(stats).view(np.uint32).reshape(-1, 6)
                assert (raw[:, 3] == 0).all()
                assert np.array_equal(raw[:, 2], stats["n_hsp"])
                assert np.array_equal(raw[:, 4:].copy().view(np.int64)[:, 0], stats["first"])
            db.close()
