"""Results larger than what is copied before the totals are known (32 MiB in the
compact layout), than the copies' buffer (64 MiB: dense results and the gapped
stage's counters and records in two copies), and than a scan's first HSP
buffer, against the oracle, bit-exactly."""
import numpy as np
import pytest

import hbseed
import test_gpu_results as small

pytestmark = pytest.mark.gpu


def test_results_in_two_copies():
    n = 1300000
    # one HSP of 40 residues in every subject, four residues before it
    res, offs = small.database(n, 44, 9500, 1)
    rows = res.reshape(n, 44)
    rows[:, 4:] = small.Q[:40]
    rows[:, :4] = hbseed.random_protein(9501, 4 * n).reshape(n, 4)
    with hbseed.Context(0) as ctx:
        found = small.check(ctx, res, offs)
    assert found >= n
    assert 32 * found > 32 << 20                      # compact
    assert 24 * n + 32 * found > 64 << 20             # dense
    assert 16 * n + 40 * found > 64 << 20             # gapped, copied again from the start
