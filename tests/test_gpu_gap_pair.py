"""The gapped extension's pair kernel (half a wavefront per subject, windows of
64 and 128 columns, 2,048 staged letters) at the sizes where it hands work to the
general kernel, bit-exact against the oracle."""
import numpy as np
import pytest

import hbseed
from test_gpu_gapped import ctx, run_both  # noqa: F401

pytestmark = pytest.mark.gpu


def pack(parts):
    offs = np.zeros(len(parts) + 1, np.uint64)
    np.cumsum([len(p) for p in parts], out=offs[1:])
    return np.concatenate(parts).astype(np.uint8), offs


def gapped_copy(seed, q, every, size):
    """q with insertions and deletions of up to `size` residues in turn."""
    rng = np.random.default_rng(seed)
    out, at, k = [], 0, 0
    while at < len(q):
        out.append(q[at:at + every])
        at += every
        n = int(rng.integers(1, size + 1))
        if k % 2:
            at += n
        else:
            out.append(hbseed.random_protein(seed * 100 + k, n))
        k += 1
    return np.concatenate(out)


@pytest.mark.parametrize("size", [2, 9, 24])
def test_gaps_move_the_window(ctx, size):  # noqa: F811
    q = hbseed.random_protein(911, 700)
    parts = [hbseed.random_protein(920 + i, 1 + i % 5) for i in range(4)]
    for i in range(40):
        parts.append(gapped_copy(930 + 50 * size + i, q[i:], 40 + i, size))
    res, offs = pack(parts)
    _, g, _, _ = run_both(ctx, hbseed.blastp_query(q), res, offs, [60])
    assert len(g)


@pytest.mark.parametrize("period", [7, 19, 41, 83])
def test_repeats_outgrow_the_window(ctx, period):  # noqa: F811
    unit = hbseed.random_protein(1000 + period, period)
    q = np.tile(unit, 400 // period + 1)[:400]
    parts = [hbseed.homolog(1100 + i, np.tile(unit, 20)[:period + 37 * i], 0.6 + 0.02 * i, i % 3)
             for i in range(1, 9)]
    res, offs = pack(parts)
    gst, _, _, _ = run_both(ctx, hbseed.blastp_query(q), res, offs, [50])
    assert gst["extensions"].sum()


@pytest.mark.parametrize("slen", [2047, 2048, 2049, 2052, 5000, 12001])
def test_subjects_around_the_staged_length(ctx, slen):  # noqa: F811
    """Homologs at the start, the middle and the end, and one of 2,600 residues
    whose alignment runs past the staged letters."""
    q = hbseed.random_protein(1200, 2600)
    parts = []
    for i in range(8):
        s = hbseed.random_protein(1210 + i, slen + i % 4)
        h = hbseed.homolog(1230 + i, q[100 * i:100 * i + 300], 0.7, 2)
        at = [0, (len(s) - len(h)) // 2, len(s) - len(h)][i % 3]
        s[at:at + len(h)] = h
        parts.append(s)
    parts.append(np.concatenate([hbseed.random_protein(1250, slen), hbseed.homolog(1251, q, 0.8, 3)]))
    res, offs = pack(parts)
    _, g, _, _ = run_both(ctx, hbseed.blastp_query(q), res, offs, [70])
    assert len(g)


@pytest.mark.parametrize("mirrored", [False, True])
def test_leading_gaps_of_the_drop_off(ctx, mirrored):  # noqa: F811
    """A short piece of the query next to a copy of it 20 to 32 diagonals away:
    the extension of the piece starts with a gap that costs about the drop-off
    (27 residues: all of it)."""
    q = hbseed.random_protein(1260, 90)
    parts = []
    for d in range(20, 33):
        for m in range(4, 10):
            for i in range(0, 40, 3):
                j = max(0, i + m - d)
                gap = j + d - i - m
                parts.append(np.concatenate([hbseed.random_protein(4 * i + m, 4), q[i:i + m],
                                             hbseed.random_protein(100 * d + i, gap), q[j:]]))
    if mirrored:
        q = q[::-1].copy()
        parts = [p[::-1].copy() for p in parts]
    res, offs = pack(parts)
    _, g, _, _ = run_both(ctx, hbseed.blastp_query(q), res, offs, [20])
    assert len(g) > len(parts)


@pytest.mark.parametrize("n", [32, 33, 64, 128, 129, 300])
def test_many_hsps_and_many_saved(ctx, n):  # noqa: F811
    q = hbseed.random_protein(1300, 300)
    parts = []
    for k in range(n):
        a = (37 * k) % 240
        parts.append(hbseed.homolog(1310 + k, q[a:a + 60], 0.9, 0))
        parts.append(hbseed.random_protein(1800 + k, 5))
    big = np.concatenate(parts)
    res, offs = pack([q[:50], big, hbseed.random_protein(1301, 77), big[:len(big) // 2]])
    gst, _, _, _ = run_both(ctx, hbseed.blastp_query(q), res, offs, [60])
    assert gst["n_hsp"].max() >= n // 2


@pytest.mark.parametrize("go,ge,x", [(11, 1, 42), (11, 1, 43), (0, 1, 20), (0, 2, 61), (10, 100, 900),
                                     (10, 101, 900), (900, 100, 8000), (900, 100, 8001),
                                     (11, 0, 38), (3, 1, 0)])
def test_parameters_around_the_rule(ctx, go, ge, x):  # noqa: F811
    q = hbseed.random_protein(1400, 350)
    res, offs = hbseed.make_db(1401, 600, plant_query=q, plant_frac=0.2)
    run_both(ctx, hbseed.blastp_query(q), res, offs, [50], go, ge, x)


def test_scores_at_the_ends_of_their_type(ctx):  # noqa: F811
    """Six frames with stop letters, subjects of one word, homologs cut at either
    end of subject and context."""
    pq = hbseed.random_protein(1500, 400)
    spec = hbseed.blastx_query(hbseed.blastx_nt(1501, 1400, pq[:150], pq[200:380]))
    parts = [pq[:3], pq[:150], pq[5:150], pq[:140], pq[200:380], pq[203:377]]
    parts += [hbseed.homolog(1510 + i, pq[200:380], 0.8, 2) for i in range(20)]
    res, offs = pack(parts)
    _, g, _, _ = run_both(ctx, spec, res, offs, [40] * len(spec.ctx_off))
    assert len(g)
