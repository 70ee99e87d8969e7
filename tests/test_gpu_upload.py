"""Loading from pageable and page-locked memory at the sizes where the upload's
chunks change, databases one after the other in the same buffers, and from
several threads, against the oracle's scan, bit-exactly."""
import threading

import numpy as np
import pytest

import hbseed
import oracle_lib

pytestmark = pytest.mark.gpu

Q = hbseed.random_protein(8980, 60)
SPEC = hbseed.blastp_query(Q, cutoff=20)
MIB = 1 << 20


@pytest.fixture(scope="module")
def ctx():
    c = hbseed.Context(0)
    yield c
    c.close()


def database(total, seed, lead=0):
    """Subjects of about 1,000 residues, `total` in all, the query at the end of
    every 97th and of the last; `lead` residues before the first."""
    lens = np.full(total // 1000, 1000, np.int64)
    lens[-1] += total - int(lens.sum())
    offs = np.zeros(len(lens) + 1, np.uint64)
    offs[1:] = np.cumsum(lens)
    res = hbseed.random_protein(seed, total + lead)
    offs += np.uint64(lead)
    for i in list(range(0, len(lens), 97)) + [len(lens) - 1]:
        e = int(offs[i + 1])
        res[e - len(Q):e] = Q
    return res, offs


def check(ctx, res, offs):
    lead = int(offs[0])
    cnt, ref = oracle_lib.OracleQuery.from_spec(SPEC).scan(res[lead:].copy(), offs - np.uint64(lead),
                                                           threads=8)
    db = hbseed.Database(ctx, res, offs)
    stats, hsps = hbseed.search(ctx, db, SPEC)
    db.close()
    assert len(ref) > 0
    assert np.array_equal(hsps.view(np.int32), ref.view(np.int32))
    assert np.array_equal(stats["lookup_hits"], cnt[:, 0])


@pytest.mark.parametrize("locked", [False, True])
@pytest.mark.parametrize("total", [4 * MIB - 1, 4 * MIB, 4 * MIB + 1, 5 * MIB, 7 * MIB - 1, 7 * MIB + 1,
                                   11 * MIB, 19 * MIB + 3])
def test_sizes(ctx, total, locked):
    res, offs = database(total, 8981 + total % 7, lead=total % 5)
    if not locked:
        check(ctx, res, offs)
        return
    with ctx.pinned(len(res)) as buf:
        buf.array[:] = res
        check(ctx, buf.array, offs)


def test_one_after_the_other(ctx):
    """Smaller and larger databases in the last one's buffers; a load that fails
    in between."""
    for k, total in enumerate([9 * MIB, 6 * MIB, 9 * MIB + 1000, 5000, 8 * MIB]):
        res, offs = database(total, 8990 + k)
        check(ctx, res, offs)
        res[-1] = 99
        with pytest.raises(hbseed.HBError):
            hbseed.Database(ctx, res, offs)


def test_volume_equals_packed(ctx):
    res, offs, _ = hbseed.sort_by_length(*hbseed.make_db(8995, 30000, plant_query=Q, plant_frac=0.05))
    n = hbseed.hdb_gpu_seqs(30000)
    vol, group_len = hbseed.hdb_pack(res, offs, n)
    assert vol.nbytes > 8 * MIB
    out = []
    for db in (hbseed.Database.from_hdb(ctx, vol, 512, 192, n, group_len),
               hbseed.Database(ctx, res[:int(offs[n])], offs[:n + 1])):
        out.append(hbseed.search(ctx, db, SPEC))
        db.close()
    assert len(out[0][1])
    for a, b in zip(out[0], out[1]):
        assert np.array_equal(a, b)


def test_threads(ctx):
    """Two contexts and two threads on one of them load and search at once."""
    other = hbseed.Context(0)
    failed = []

    def run(c, seed):
        try:
            for k in range(3):
                check(c, *database(5 * MIB + 4096 * k, seed + k))
        except BaseException as e:   # noqa: BLE001
            failed.append(e)

    th = [threading.Thread(target=run, args=a) for a in ((ctx, 8900), (ctx, 8910), (other, 8920))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    other.close()
    assert not failed, failed
