"""Subjects that a pass of the gapped extension leaves to the next one go on
where they were left: after no, one, the most and more gapped HSPs than a pass
keeps, from the pair kernel to the general one and from there to the wide pass,
bit-exact against the oracle."""
import numpy as np
import pytest

import hbseed
from test_gpu_gap_pair import pack
from test_gpu_gapped import ctx, run_both  # noqa: F401

pytestmark = pytest.mark.gpu

UNIQUE = hbseed.random_protein(9700, 400)


def pieces(seed, n):
    """n homologs of pieces of the query, best first, apart from each other."""
    out = []
    for k in range(n):
        a = (37 * k) % 330
        out.append(hbseed.homolog(seed + k, UNIQUE[a:a + 70], 0.95, 0))
        out.append(hbseed.random_protein(seed + 500 + k, 6))
    return out


@pytest.mark.parametrize("before", [0, 1, 31, 32, 33, 45])
@pytest.mark.parametrize("period,x", [(41, 38), (7, 42)])
def test_left_after(ctx, before, period, x):  # noqa: F811
    unit = hbseed.random_protein(9710 + period, period)
    rep = np.tile(unit, 700 // period)
    query = np.concatenate([UNIQUE, hbseed.random_protein(9720, 30), rep])
    parts = []
    for i in range(6):
        bent = hbseed.homolog(9730 + i, np.tile(unit, (150 + 60 * i) // period), 0.62, 2)
        s = pieces(9740 + 1000 * i, before)
        at = (len(s) // 2) * (i % 2)     # the repeat in the middle or at the start
        parts.append(np.concatenate(s[:at] + [bent] + s[at:]))
    res, offs = pack(parts)
    gst, g, _, _ = run_both(ctx, hbseed.blastp_query(query), res, offs, [45], x_dropoff=x)
    assert gst["n_hsp"].max() >= before


def test_two_contexts(ctx):  # noqa: F811
    """The list of saved HSPs keeps their contexts."""
    spec = hbseed.blastx_query(hbseed.blastx_nt(9760, 1800, UNIQUE[:250], UNIQUE[100:380]))
    parts = []
    for i in range(4):
        s = pieces(9770 + 1000 * i, 30 + 4 * i)
        parts.append(np.concatenate(s + [UNIQUE[:250], UNIQUE[100:380]]))
    res, offs = pack(parts)
    gst, _, _, _ = run_both(ctx, spec, res, offs, [40] * len(spec.ctx_off))
    assert gst["n_hsp"].max() > 32
