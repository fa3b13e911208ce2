"""The one-grain refinement's block sums: numbers of blocks around the rounds
in which the last launch takes them in, and its largest."""

import numpy as np
import pytest
import torch

from imaged11_amd import cImageD11

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng", [1, 1024, 1025, 127 * 1024 + 1, 128 * 1024, 128 * 1024 + 1,
                                256 * 1024 + 3, 1024 * 1024, 1024 * 1024 + 7])
@pytest.mark.parametrize("assigned", [False, True])
def test_block_sums(dev, orc, ng, assigned):
    # g a multiple of 1/8 and h an integer multiple of it: every sum is exact
    # in 53 bits (|terms| <= 64, a multiple of 1/64, at most 2^20 + 7 of them),
    # so that the order of the additions doesn't matter and the bits are the
    # oracle's
    rng = np.random.default_rng(ng)
    gv = rng.integers(-8, 9, (ng, 3)) / 8.0
    u = np.array([[8.0, 0, 0], [0, 8.0, 0], [0, 0, 8.0]])
    ug, uo = u.copy(), u.copy()
    g = torch.as_tensor(gv, device=dev)
    if assigned:
        lab = rng.integers(0, 3, ng).astype(np.int32)
        got = cImageD11.refine_assigned(ug, g, torch.as_tensor(lab, device=dev), 1)
        want = orc.refine_assigned(uo, gv, lab, 1)
    else:
        got = cImageD11.score_and_refine(ug, g, 0.05)
        want = orc.score_and_refine(uo, gv, 0.05)
    assert got[0] == want[0]
    assert got[1] == want[1]
    assert np.array_equal(ug, uo)
