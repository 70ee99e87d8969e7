"""Loading a database: record order and the residue copy at the edges of the
loader's steps (16-byte pieces, 16 KB blocks, 4,096 subjects, lengths past the
counted ones), against the oracle's scan, bit-exactly; a residue that is no
code is found wherever it stands."""
import numpy as np
import pytest

import hbseed
import oracle_lib

pytestmark = pytest.mark.gpu

Q = hbseed.random_protein(9980, 60)


@pytest.fixture(scope="module")
def ctx():
    c = hbseed.Context(0)
    yield c
    c.close()


def database(lens, seed):
    """Random residues, each subject with as much of the query as fits."""
    lens = np.asarray(lens, np.int64)
    offs = np.zeros(len(lens) + 1, np.uint64)
    offs[1:] = np.cumsum(lens)
    res = hbseed.random_protein(seed, max(int(lens.sum()), 1))[:int(lens.sum())]
    for i, n in enumerate(lens):
        k = min(int(n), len(Q))
        res[int(offs[i]) + int(n) - k:int(offs[i]) + int(n)] = Q[:k]
    return res, offs


CASES = {
    "one": [37],
    "short": list(range(0, 40)) * 3,
    "empty": [0] * 100 + [50] + [0] * 5000,
    "equal": [45] * 4097,
    "4095": list(np.random.default_rng(1).integers(0, 90, 4095)),
    "4096": list(np.random.default_rng(2).integers(0, 90, 4096)),
    "block": [16384, 16383, 16385, 32768, 15, 16, 17, 1, 0],
    "long": [65535, 65536, 65537, 70000, 70000, 100, 3, 140000, 65536],
}


@pytest.mark.parametrize("name", CASES)
def test_order_and_copy(ctx, name):
    res, offs = database(CASES[name], 9981)
    spec = hbseed.blastp_query(Q, cutoff=10)
    cnt, ref = oracle_lib.OracleQuery.from_spec(spec).scan(res, offs, threads=8)
    db = hbseed.Database(ctx, res, offs)
    stats, hsps = hbseed.search(ctx, db, spec)
    assert len(ref) > 0
    assert np.array_equal(hsps.view(np.int32), ref.view(np.int32))
    assert np.array_equal(stats["lookup_hits"], cnt[:, 0])
    assert np.array_equal(stats["n_hsp"], cnt[:, 2])
    db.close()


@pytest.mark.parametrize("code", [28, 127, 128, 255])
@pytest.mark.parametrize("lens,at", [([5], 4), ([5, 40], 0), ([5, 40], 44), ([16, 16], 16),
                                     ([40000], 16384), ([40000], 39999), ([3, 0, 17, 2], 19)])
def test_residue_check(ctx, lens, at, code):
    res, offs = database(lens, 9982)
    hbseed.Database(ctx, res, offs).close()
    res[at] = code
    with pytest.raises(hbseed.HBError) as e:
        hbseed.Database(ctx, res, offs)
    assert "RESIDUE" in str(e.value).upper() or e.value.code == hbseed.HB_ERR_RESIDUE
