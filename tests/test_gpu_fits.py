"""The per-task fits at row counts around the lanes that share a task."""
import numpy as np
import pytest
import torch

from imaged11_amd import point_by_point as PP

pytestmark = pytest.mark.gpu

ROWS = [0, 1, 2, 3, 5, 6, 7, 15, 16, 17, 31, 32, 33, 47, 64, 65, 200, 1000]


@pytest.mark.parametrize("tasks", [1, 3, 4, 5, len(ROWS)])
def test_fits_equal_lstsq(dev, tasks):
    """Random designs: the solution is within eps times the condition number
    (< 1e3 here, or a rank below full with the minimum-norm solution)."""
    rng = np.random.default_rng(tasks)
    rows = ROWS[-tasks:]
    off = np.concatenate([[0], np.cumsum(rows)]).astype(np.int64)
    T = lambda a, dt=torch.float64: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=dev)
    for nc, nr in ((6, 1), (3, 3)):
        design = rng.normal(size=(off[-1], nc + nr))
        # the product's two row layouts: (M, strain) and (g, hkl)
        on = torch.ones(tasks, dtype=torch.bool, device=dev)
        if nc == 6:
            got = PP.strain_fit(T(design), T(off, torch.int64), on).cpu().numpy()
        else:
            ubis = T(np.broadcast_to(np.eye(3), (tasks, 3, 3)))
            fit, rank, _, _, _ = PP.ubi_fit(T(design), T(off, torch.int64), on, ubis, np.eye(3))
            got, rank = fit.cpu().numpy(), rank.cpu().numpy()
        for t in range(tasks):
            d = design[off[t]:off[t + 1]]
            if len(d) == 0:
                want, r = np.zeros((nc, nr)), 0
            else:
                want, _, r, sv = np.linalg.lstsq(d[:, :nc], d[:, nc:], rcond=None)
                if sv.min() < 1e-3 * sv.max():
                    continue
            if nc == 6:
                np.testing.assert_allclose(got[t], want[:, 0], rtol=0, atol=1e-11)
            else:
                np.testing.assert_allclose(got[t], want.T, rtol=0, atol=1e-11)
                assert rank[t] == r
