"""score_and_assign on host arrays: in place in pinned memory up to 1 MiB of
them, by copies to the device beyond; the oracle's counts, labels and drlv2."""

import numpy as np
import pytest

from imaged11_amd import cImageD11

pytestmark = pytest.mark.gpu

EDGE = (1 << 20) // 36  # the most peaks in pinned memory


@pytest.mark.parametrize("ng", [0, 1, 511, 512, 513, 20000, EDGE, EDGE + 1, 60000])
def test_host_score_and_assign(dev, orc, ng):
    rng = np.random.default_rng(ng)
    u = 4.0 * np.linalg.qr(rng.normal(size=(3, 3)))[0]
    gv = (rng.integers(-5, 6, (ng, 3)) + rng.normal(scale=0.03, size=(ng, 3))) @ np.linalg.inv(u).T
    gv[::31] = np.nan
    d, lab = rng.uniform(0, 0.01, ng), rng.integers(-1, 4, ng).astype(np.int32)
    do, lo = d.copy(), lab.copy()
    for label in (2, 7, 2):  # wins, ties with itself, and a label taken away again
        got = cImageD11.score_and_assign(u, gv, 0.05, d, lab, label)
        want = orc.score_and_assign(u, gv, 0.05, do, lo, label)
        assert got == want
        assert np.array_equal(lab, lo) and np.array_equal(d, do)
        u = u * (1 + 1e-4)
