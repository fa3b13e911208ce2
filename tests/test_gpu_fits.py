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


@pytest.mark.parametrize("lanes", [1, 4, 16])
@pytest.mark.parametrize("cond", [10.0, 1e5, 1e10])
def test_fits_are_backward_stable(dev, lanes, cond):
    """Every lane count, designs of any condition: the solution is that of a
    design within a few (rows + columns) roundings, so its gradient is below
    10 (m + n) eps |A| (|r| + |A| |x|), in extended precision."""
    rng = np.random.default_rng(7)
    off = np.concatenate([[0], np.cumsum([r for r in ROWS if r >= 6])]).astype(np.int64)
    tasks = len(off) - 1
    T = lambda a, dt=torch.float64: torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=dev)
    on = torch.ones(tasks, dtype=torch.bool, device=dev)
    for nc, nr in ((6, 1), (3, 3)):
        q = np.linalg.qr(rng.normal(size=(nc, nc)))[0] * np.geomspace(1.0, 1.0 / cond, nc)
        design = rng.normal(size=(off[-1], nc + nr))
        design[:, :nc] = design[:, :nc] @ q.T
        if nc == 6:
            got = PP.strain_fit(T(design), T(off, torch.int64), on, lanes=lanes)[:, :, None]
        else:
            ubis = torch.eye(3, dtype=torch.float64, device=dev).repeat(tasks, 1, 1)
            fit, rank, _, _, _ = PP.ubi_fit(T(design), T(off, torch.int64), on, ubis, np.eye(3),
                                            lanes=lanes)
            assert (rank == 3).all()
            got = fit.transpose(1, 2)
        got = got.cpu().numpy().astype(np.longdouble)
        for t in range(tasks):
            d = design[off[t]:off[t + 1]].astype(np.longdouble)
            A, m = d[:, :nc], len(d)
            size = np.linalg.norm(A.astype(float), 2)
            for c in range(nr):
                r = A @ got[t][:, c] - d[:, nc + c]
                norm = lambda v: float(np.sqrt((v * v).sum()))
                assert norm(A.T @ r) <= 10 * (m + nc) * 2.0 ** -52 * size * (
                    norm(r) + size * norm(got[t][:, c]))


@pytest.mark.parametrize("T,rows", [(1500, 24), (1501, 24), (1501, 23), (6000, 120), (6001, 120),
                                    (12288, 24), (12289, 24), (70000, 6)])
def test_fits_of_many_tasks(dev, T, rows):
    """Both sides of the lines of fit_lanes: the same as with one lane a task,
    to the designs' condition (below 100)."""
    want = {(1500, 24): 16, (6000, 120): 16, (1501, 24): 4, (6001, 120): 4, (12288, 24): 4}
    assert PP.fit_lanes(T, T * rows) == want.get((T, rows), 1)
    assert PP.fit_lanes(32768, 32768 * 150) == 4 and PP.fit_lanes(32769, 32769 * 150) == 1
    g = torch.Generator(device="cuda")
    g.manual_seed(T)
    off = torch.arange(T + 1, device=dev) * rows
    on = torch.arange(T, device=dev) % 7 != 3
    M = torch.randn((T * rows, 6), generator=g, dtype=torch.float64, device=dev)
    M += 3.0 * torch.eye(6, dtype=torch.float64, device=dev).repeat(-(-T * rows // 6), 1)[:T * rows]
    D = torch.cat([M, torch.randn((T * rows, 1), generator=g, dtype=torch.float64, device=dev)], 1)
    a, b = PP.strain_fit(D, off, on), PP.strain_fit(D, off, on, lanes=1)
    assert torch.equal(torch.isnan(a), ~on[:, None].expand(T, 6))
    s = torch.linalg.svdvals(M.view(T, rows, 6))
    scale = (s[:, :1] / s[:, -1:]) ** 2 * (b.norm(dim=1, keepdim=True) + 1.0)
    assert ((a - b).abs() <= 20 * (rows + 6) * 2.0 ** -52 * scale)[on].all()
