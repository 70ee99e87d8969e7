"""Queries around the lengths whose LDS lets five workgroups into a CU, against
databases around the size from which 20 wavefronts per CU scan them, in one and
two contexts and with the state forced either way, bit-exact against the
oracle."""
import numpy as np
import pytest

import hbseed
import oracle_lib

pytestmark = pytest.mark.gpu

SHARE = 256 * 16 * 4096   # residues from which 16 wavefronts per CU have their share


@pytest.fixture(scope="module")
def setup():
    ctx = hbseed.Context(0)
    q = hbseed.random_protein(9800, 400)
    res, offs = hbseed.make_db(9801, 60000, plant_query=q, plant_frac=0.05)
    assert int(offs[-1]) > SHARE
    n_few = int(np.searchsorted(offs, SHARE)) - 1      # the last size below it
    dbs = {}
    for name, n in (("below", n_few), ("at", n_few + 1), ("above", len(offs) - 1)):
        r, o = res[:int(offs[n])].copy(), offs[:n + 1].copy()
        if name == "at":   # exactly the share
            r, o = res[:SHARE].copy(), np.append(offs[:n], np.uint64(SHARE))
        dbs[name] = (hbseed.Database(ctx, r, o), r, o)
    yield ctx, q, dbs
    for db, _, _ in dbs.values():
        db.close()
    ctx.close()


@pytest.mark.parametrize("size", ["below", "at", "above"])
@pytest.mark.parametrize("n", [5, 88, 89, 152, 153, 200])
def test_lengths(setup, size, n):
    ctx, q, dbs = setup
    db, res, offs = dbs[size]
    spec = hbseed.blastp_query(q[:n].copy(), cutoff=25)
    cnt, ref = oracle_lib.OracleQuery.from_spec(spec).scan(res, offs, threads=8)
    stats, hsps = hbseed.search(ctx, db, spec)
    assert len(ref) > 0 or n < 25
    assert np.array_equal(hsps.view(np.int32), ref.view(np.int32))
    for i, f in enumerate(("lookup_hits", "extensions", "n_hsp")):
        assert np.array_equal(stats[f], cnt[:, i])


@pytest.mark.parametrize("mode", [hbseed.STATE_GLOBAL, hbseed.STATE_LDS])
def test_six_frames(setup, mode):
    ctx, q, dbs = setup
    db, res, offs = dbs["above"]
    spec = hbseed.blastx_query(hbseed.blastx_nt(9810, 72, q[:10], q[20:30]))
    assert len(spec.seq) <= 152
    cnt, ref = oracle_lib.OracleQuery.from_spec(spec).scan(res, offs, threads=8)
    query = hbseed.Query(ctx, spec)
    query.set_state_mode(mode)
    query.set_reset_interval(20000)
    scan = hbseed.Scan(ctx, db, query)
    stats, hsps = scan.results()
    scan.close()
    query.close()
    assert np.array_equal(hsps.view(np.int32), ref.view(np.int32))
    assert np.array_equal(stats["lookup_hits"], cnt[:, 0])
