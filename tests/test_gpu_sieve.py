"""The matrix-core sieve against the reference arithmetic, at the sizes and
values where its tiles, ranges and queues can go wrong."""
import numpy as np
import pytest
import torch

from imaged11_amd import batched, simulate

pytestmark = pytest.mark.gpu


def T(a, dev, dt=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device=dev)


def make(K, N, seed, cell=(3.0, 9.0), gmax=1.6, own=0.3):
    """K UBIs and N g-vectors, a share `own` of them near-lattice points of
    the grains (so that hits of every distance around tol occur)."""
    rng = np.random.default_rng(seed)
    ub = simulate.random_rotations(K, rng) / rng.uniform(*cell, size=(K, 3))[:, None, :]
    gv = rng.uniform(-gmax, gmax, size=(N, 3))
    m = int(own * N)
    g = rng.integers(0, K, m)
    hkl = np.einsum("nij,nj->ni", np.linalg.inv(ub)[g], gv[:m])
    gv[:m] = np.einsum("nij,nj->ni", ub[g], np.round(hkl) + rng.normal(scale=0.04, size=(m, 3)))
    return np.linalg.inv(ub), gv


@pytest.mark.parametrize("K,N", [(1, 1), (1, 5000), (31, 127), (32, 128), (33, 129), (64, 511),
                                 (65, 513), (129, 4097), (2049, 700), (3, 100001)])
@pytest.mark.parametrize("tol", [0.003, 0.05, 0.1])
def test_counts_at_tile_edges(dev, orc, K, N, tol):
    ubi, gv = make(K, N, K + N)
    got = batched.score_sieve(T(ubi, dev), T(gv, dev), tol)
    assert np.array_equal(got.cpu().numpy(), orc.score_many(ubi, gv, tol))


# the largest row sum of |u| times max |g|: inside the narrow range, across
# its end, the wide range, across its end, beyond; |u| and |g| past f16
@pytest.mark.parametrize("cell,gmax", [((10.0, 20.0), 1.6), ((20.0, 60.0), 1.6),
                                       ((200.0, 320.0), 1.6), ((300.0, 900.0), 1.6),
                                       ((900.0, 2000.0), 0.01), ((0.05, 0.2), 40.0),
                                       ((1e-4, 2e-4), 1e4), ((2e6, 5e6), 1e-6)])
def test_counts_over_the_ranges_of_the_accumulator(dev, orc, cell, gmax):
    ubi, gv = make(70, 3000, 5, cell=cell, gmax=gmax)
    for tol in (0.02, 0.1):
        got = batched.score_sieve(T(ubi, dev), T(gv, dev), tol)
        want = orc.score_many(ubi, gv, tol)
        assert want.sum() > 0
        assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("tol", [0.2, 0.45, 0.5, 1.0])
def test_counts_at_tolerances_the_queues_overflow(dev, orc, tol):
    ubi, gv = make(40, 2000, 9)
    got = batched.score_sieve(T(ubi, dev), T(gv, dev), tol)
    assert np.array_equal(got.cpu().numpy(), orc.score_many(ubi, gv, tol))


def test_special_values(dev, orc):
    """NaN, infinite, zero and huge rows and UBIs beside ordinary ones."""
    ubi, gv = make(40, 1000, 11)
    bad = [np.nan, np.inf, -np.inf, 1e300, 1e-310, 0.0]
    for i, v in enumerate(bad):
        gv[17 * i + 3, i % 3] = v
        gv[17 * i + 5] = v
        ubi[2 * i, i % 3, (i + 1) % 3] = v
        ubi[2 * i + 13] = v
    for tol in (0.05, 0.0, float("nan")):
        got = batched.score_sieve(T(ubi, dev), T(gv, dev), tol)
        assert np.array_equal(got.cpu().numpy(), orc.score_many(ubi, gv, tol))


def test_pairs_on_the_tolerance(dev, orc):
    """Pairs whose distance straddles tol by 1e-17 .. 1e-3 in one row, with
    the others zero: the sieve may not drop one the reference counts."""
    a, tol = 4.0, 0.05
    d = np.array([tol * (1 + s * 10.0 ** -e) for s in (-1, 1) for e in range(3, 17)])
    hkl = np.array([[h, k, l] for h in range(-6, 7, 3) for k in (-5, 0, 4) for l in (-3, 2)],
                   float)
    gv = []
    for row in range(3):
        for s in (-1, 1):
            h = np.repeat(hkl, len(d), 0)
            h[:, row] += s * np.tile(d, len(hkl))
            gv.append(h / a)
    gv = np.concatenate(gv)
    rng = np.random.default_rng(3)
    U = simulate.random_rotations(20, rng)
    for k in range(20):
        g = gv @ U[k].T
        ubi = np.concatenate([(a * U[k].T)[None], make(33, 1, k)[0]])
        got = batched.score_sieve(T(ubi, dev), T(g, dev), tol)
        want = orc.score_many(ubi, g, tol)
        assert 0 < want[0] < len(g)
        assert np.array_equal(got.cpu().numpy(), want)


def test_graph_replays_equal_the_eager_counts(dev):
    """Captured and replayed with eager work in between; the workspace is
    the capture's own."""
    ubi, gv = make(100, 5000, 21)
    u, g = T(ubi, dev), T(gv, dev)
    out = torch.empty(100, dtype=torch.int32, device=dev)
    batched.score_sieve(u, g, 0.05, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        batched.score_sieve(u, g, 0.05, out=out)
    for rep in range(4):
        g.copy_(T(make(100, 5000, 30 + rep)[1], dev))
        out.fill_(-7)
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        assert torch.equal(got, batched.score_many(u, g, 0.05, exact=True))
