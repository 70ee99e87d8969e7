"""hb_scan_noalloc with queries whose diagonals are split into classes: the
counters of a subject are then added up over its classes, over whatever the
caller's array held."""
import pytest

import hbseed
import test_zz_no_alloc as plain

pytestmark = pytest.mark.gpu


class Hip(plain.Hip):
    def fill(self, p, byte, n):
        """Done when it returns: the scan's stream does not wait for the null
        stream, and here the counters are cleared before anything else."""
        super().fill(p, byte, n)
        self.sync()


@pytest.mark.parametrize("n", [1500, 3000, 8001, 24000])
def test_split_diagonals(n):
    spec = hbseed.blastp_query(hbseed.random_protein(9600 + n, n))
    res, offs = hbseed.make_db(9601 + n, 4000, plant_query=spec.seq[:3000], plant_frac=0.2)
    hip = Hip()
    with hbseed.Context(0) as ctx:
        db = hbseed.Database(ctx, res, offs)
        q = hbseed.Query(ctx, spec)
        stats, hsps, _ = plain.reference(ctx, db, q)
        for _ in range(2):
            recs, cnt = plain.noalloc(ctx, hip, db, q, len(offs) - 1, len(hsps) + 1000)
            plain.check(stats, hsps, recs, cnt)
        q.close()
        db.close()
