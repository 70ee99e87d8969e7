"""Lookup tables built on the device equal the oracle's, entry by entry:
query lengths around the steps of the builder (64 words, 256 words), tables
with far more entries per word than usual and thresholds past the range of
three scores, several contexts, and matrices of extreme scores."""
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


def check(ctx, spec, **kw):
    q = hbseed.Query(ctx, spec, **kw)
    start, ent = q.lut()
    q.close()
    ostart, oent = oracle_lib.OracleQuery.from_spec(spec, **kw).lut_arrays()
    assert np.array_equal(start, ostart)
    assert np.array_equal(ent, oent)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 63, 66, 67, 255, 256, 257, 258, 259, 515, 4000])
def test_query_lengths(ctx, n):
    check(ctx, hbseed.blastp_query(hbseed.random_protein(9500 + n, n)))


@pytest.mark.parametrize("threshold", [-2**31, -1000, 0, 1, 7, 33, 34, 1000, 2**31 - 1])
@pytest.mark.parametrize("n", [5, 130])
def test_thresholds(ctx, n, threshold):
    # from every word of the alphabet in every cell to the exact words only
    check(ctx, hbseed.blastp_query(hbseed.random_protein(9600 + n, n)), threshold=threshold)


@pytest.mark.parametrize("letter", [20, 0, 21])   # W, gap, X
def test_one_letter(ctx, letter):
    check(ctx, hbseed.blastp_query(np.full(300, letter, np.uint8)))


def test_contexts_and_mask(ctx):
    seq = hbseed.random_protein(9700, 400)
    mask = np.zeros(400, np.uint8)
    mask[[10, 50, 51, 52, 300]] = 1
    spec = hbseed.QuerySpec(seq, [0, 2, 70, 71, 390], [2, 60, 0, 300, 10], lut_mask=mask)
    check(ctx, spec)


@pytest.mark.parametrize("seed", [1, 2])
def test_extreme_matrix(ctx, seed):
    m = np.random.default_rng(seed).choice([-128, -127, 0, 126, 127], (28, 28)).astype(np.int8)
    for t in (-384, -383, 11, 380, 381):
        check(ctx, hbseed.blastp_query(hbseed.random_protein(9800 + seed, 90)), matrix=m, threshold=t)
