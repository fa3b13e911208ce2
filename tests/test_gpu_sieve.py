"""The matrix-core sieve against the reference arithmetic, at the sizes and
values where its tiles, ranges and queues can go wrong."""
import numpy as np
import pytest
import torch

from imaged11_amd import _lib, batched, simulate

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


# ---- assignment ------------------------------------------------------------


def scan_inputs(K, N, seed, dist=150000.0, t=200.0, cell=(3.0, 9.0), wvln=0.2):
    rng = np.random.default_rng(seed)
    ubi = np.linalg.inv(simulate.random_rotations(K, rng) /
                        rng.uniform(*cell, size=(K, 3))[:, None, :])
    trans = rng.uniform(-t, t, size=(K, 3)) if t else np.zeros((K, 3))
    ang = rng.uniform(0, 0.35, N)
    eta = rng.uniform(0, 2 * np.pi, N)
    xl = dist / np.cos(ang)[:, None] * np.stack([np.cos(ang), np.sin(ang) * np.cos(eta),
                                                 np.sin(ang) * np.sin(eta)], 1)
    om = rng.uniform(-np.pi, np.pi, N)
    return ubi, trans, xl, np.sin(om), np.cos(om), wvln, rng


def check_scan(dev, orc, ubi, trans, xl, so, co, wvln, tol, d0, l0, mat=None):
    """gv_assign_many with default labels (the sieve) against the oracle's loop."""
    K = len(ubi)
    mat = np.eye(3) if mat is None else mat
    d, lab = d0.copy(), l0.copy()
    want = orc.gv_assign_many(xl, so, co, mat, wvln, ubi, trans, np.arange(K), tol, d, lab)
    dd, ll = T(d0, dev), T(l0, dev, torch.int32)
    assert batched.assign_mfma_pays(K, len(xl), tol)
    got = batched.gv_assign_many(T(xl, dev), T(so, dev), T(co, dev), wvln, T(ubi, dev),
                                 T(trans, dev), tol, dd, ll, mat=mat)
    assert np.array_equal(got.cpu().numpy(), want)
    assert np.array_equal(ll.cpu().numpy(), lab)
    assert np.array_equal(dd.cpu().numpy().view(np.int64), d.view(np.int64))
    return want


@pytest.mark.parametrize("K,N", [(16, 1), (16, 31), (31, 32), (32, 33), (33, 127), (64, 129),
                                 (65, 511), (2049, 600), (20, 140000), (17, 270001)])
def test_scan_at_tile_edges(dev, orc, K, N):
    ubi, trans, xl, so, co, w, rng = scan_inputs(K, N, K + N)
    check_scan(dev, orc, ubi, trans, xl, so, co, w, 0.1, np.ones(N), np.full(N, -1, np.int32))


# positions from none to as large as the detector distance (micron and other
# units), so that tiles are sieved, sieved with a wide radius, or not at all
@pytest.mark.parametrize("dist,t", [(150000.0, 0.0), (150000.0, 1000.0), (150000.0, 6000.0),
                                    (150000.0, 20000.0), (8000.0, 300.0), (5000.0, 2600.0),
                                    (150.0, 0.2), (0.15, 2e-4), (150000.0, 200000.0)])
@pytest.mark.parametrize("cell", [(3.0, 9.0), (20.0, 45.0), (300.0, 1200.0)])
def test_scan_over_positions_and_cells(dev, orc, dist, t, cell):
    ubi, trans, xl, so, co, w, rng = scan_inputs(100, 3000, 4, dist=dist, t=t, cell=cell)
    mat = orc.wedge_chi_matrix(1.5, -2.0).reshape(3, 3)
    want = check_scan(dev, orc, ubi, trans, xl, so, co, w, 0.1, np.ones(3000),
                      np.full(3000, -1, np.int32), mat)
    assert want.sum() > 300


# lengths, cells and wavelengths towards the ends of f32 and past them; one
# detector distance of positions beyond |a| / 2
@pytest.mark.parametrize("dist,t,cell,wvln", [(8000.0, 500.0, (3.0, 9.0), 0.2),
                                              (8000.0, 500.0, (3e2, 9e3), 0.2),
                                              (8000.0, 500.0, (3e4, 9e4), 0.2),
                                              (8e-9, 5e-10, (3.0, 9.0), 0.2),
                                              (8e-14, 5e-15, (3.0, 9.0), 0.2),
                                              (8e12, 5e11, (3.0, 9.0), 0.2),
                                              (8e17, 5e16, (3.0, 9.0), 0.2),
                                              (8000.0, 500.0, (3e-15, 9e-15), 2e-16),
                                              (8000.0, 500.0, (3e20, 9e20), 2e19),
                                              (8000.0, 6000.0, (3.0, 9.0), 0.2)])
@pytest.mark.parametrize("K,N", [(33, 130), (100, 3001), (40, 140001)])
def test_scan_tiles_in_f32(dev, orc, dist, t, cell, wvln, K, N):
    ubi, trans, xl, so, co, w, rng = scan_inputs(K, N, K, dist=dist, t=t, cell=cell, wvln=wvln)
    l0 = rng.integers(-2, K + 2, N).astype(np.int32)
    want = check_scan(dev, orc, ubi, trans, xl, so, co, w, 0.1, np.full(N, 2.0), l0)
    assert want.sum() > 0


@pytest.mark.parametrize("dist,t", [(150000.0, 200.0), (8000.0, 500.0)])
def test_scan_of_grains_far_off(dev, orc, dist, t):
    """One, then a third of the grains far from the others (by 0.4 and by 3
    detector distances): tiles of both kinds in one wave."""
    K, N = 170, 4000
    ubi, trans, xl, so, co, w, rng = scan_inputs(K, N, 5, dist=dist, t=t)
    for far in (np.array([77]), np.arange(0, K, 3)):
        for by in (0.4, 3.0):
            tr = trans.copy()
            tr[far, 1] = by * dist
            check_scan(dev, orc, ubi, tr, xl, so, co, w, 0.1, np.full(N, 2.0),
                       np.full(N, -1, np.int32))


@pytest.mark.parametrize("dist", [150000.0, 8000.0])
def test_scan_nonfinite_values_on_both_routes(dev, orc, dist):
    """Values that are not finite without a huge one beside them."""
    K, N = 96, 2000
    ubi, trans, xl, so, co, w, rng = scan_inputs(K, N, 9, dist=dist, t=500.0)
    for i, v in enumerate((np.nan, np.inf, -np.inf)):
        xl[200 * i + 7, i] = v
        so[200 * i + 60] = co[200 * i + 77] = v
        ubi[7 * i, i] = v
        ubi[7 * i + 1, i, 0] = v
        trans[7 * i + 2, i] = v
        trans[7 * i + 3] = v
    want = check_scan(dev, orc, ubi, trans, xl, so, co, w, 0.1, np.full(N, 2.0),
                      rng.integers(-2, K + 2, N).astype(np.int32))
    assert want.sum() > 0


@pytest.mark.parametrize("scale", [1.0, 300.0, 1e6])
def test_assignment_nonfinite_values(dev, orc, scale):
    """The same for g-vectors given: on the matrix cores, in f32, settled."""
    ubi, gv = nonfinite_inputs()
    ubi, K, N = ubi * scale, len(ubi), len(gv)
    rng = np.random.default_rng(1)
    d0, l0 = rng.uniform(0, 0.02, N), rng.integers(-2, K + 2, N).astype(np.int32)
    d, lab = d0.copy(), l0.copy()
    want = orc.assign_many(ubi, np.arange(K), gv, 0.1, d, lab)
    dd, ll = T(d0, dev), T(l0, dev, torch.int32)
    got = batched.assign_many(T(ubi, dev), T(gv, dev), 0.1, dd, ll)
    assert want.sum() > 0 and np.array_equal(got.cpu().numpy(), want)
    assert np.array_equal(ll.cpu().numpy(), lab)
    assert np.array_equal(dd.cpu().numpy().view(np.int64), d.view(np.int64))


def test_scan_from_other_states(dev, orc):
    """Labels of the grains and others, current drlv2 anywhere in reach,
    repeated grains, peaks and grains with special values, a peak at the
    origin."""
    K, N = 150, 5000
    ubi, trans, xl, so, co, w, rng = scan_inputs(K, N, 8)
    ubi[70:90], trans[70:90] = ubi[50:70], trans[50:70]  # equal drlv2: the first keeps the peak
    for i, v in enumerate([np.nan, np.inf, 1e300, 0.0]):
        xl[11 * i] = v
        xl[11 * i + 3, i % 3] = v
        ubi[5 * i, 1, 2] = v
        trans[5 * i + 40, i % 3] = v
        so[11 * i + 5] = v
    l0 = rng.integers(-3, K + 5, N).astype(np.int32)
    d0 = rng.uniform(0.0, 0.02, N)
    d0[::13] = np.nan
    d0[1::13] = np.inf
    check_scan(dev, orc, ubi, trans, xl, so, co, w, 0.1, d0, l0)


@pytest.mark.parametrize("tol", [0.001, 0.05, 0.1])
@pytest.mark.parametrize("K,N", [(16, 1), (33, 129), (300, 20001), (2100, 300)])
def test_assignment_of_gvectors(dev, orc, K, N, tol):
    ubi, gv = make(K, N, K)
    rng = np.random.default_rng(K)
    for d0, l0 in ((np.full(N, 2.0), np.full(N, -1, np.int32)),
                   (rng.uniform(0, 0.02, N), rng.integers(-2, K + 2, N).astype(np.int32))):
        d, lab = d0.copy(), l0.copy()
        want = orc.assign_many(ubi, np.arange(K), gv, tol, d, lab)
        dd, ll = T(d0, dev), T(l0, dev, torch.int32)
        got = batched.assign_many(T(ubi, dev), T(gv, dev), tol, dd, ll)
        assert np.array_equal(got.cpu().numpy(), want)
        assert np.array_equal(ll.cpu().numpy(), lab)
        assert np.array_equal(dd.cpu().numpy().view(np.int64), d.view(np.int64))


@pytest.mark.parametrize("K", [19, 20, 63, 64, 65])
@pytest.mark.parametrize("N", [300000, 300001, 131072, 5000])
def test_assignment_of_few_grains(dev, K, N):
    """Counts in LDS up to 64 grains, and the sizes that leave them to the
    FP64 loop, against the reference arithmetic."""
    ubi, gv = make(K, N, K, own=0.8)
    u, g = T(ubi, dev), T(gv, dev)
    d = [torch.full((N,), 2.0, dtype=torch.float64, device=dev) for _ in range(2)]
    lab = [torch.full((N,), -1, dtype=torch.int32, device=dev) for _ in range(2)]
    n = [batched.assign_many(u, g, 0.1, d[i], lab[i], exact=i == 1) for i in range(2)]
    assert n[1].sum().item() > N / 4
    for a, b in (n, d, lab):
        assert torch.equal(a, b)


@pytest.mark.parametrize("cell,gmax", [((20.0, 60.0), 1.6), ((300.0, 900.0), 1.6),
                                       ((0.05, 0.2), 40.0)])
def test_assignment_over_the_ranges_of_the_accumulator(dev, orc, cell, gmax):
    ubi, gv = make(90, 2000, 6, cell=cell, gmax=gmax)
    d, lab = np.ones(2000), np.full(2000, -1, np.int32)
    want = orc.assign_many(ubi, np.arange(90), gv, 0.1, d, lab)
    dd, ll = T(np.ones(2000), dev), T(np.full(2000, -1), dev, torch.int32)
    got = batched.assign_many(T(ubi, dev), T(gv, dev), 0.1, dd, ll)
    assert want.sum() > 0 and np.array_equal(got.cpu().numpy(), want)
    assert np.array_equal(ll.cpu().numpy(), lab)
    assert np.array_equal(dd.cpu().numpy().view(np.int64), d.view(np.int64))


@pytest.mark.parametrize("K,N", [(8, 2000003), (700, 30001), (2100, 8000)])
@pytest.mark.parametrize("tol", [0.02, 0.1])
def test_selected_lists(dev, K, N, tol):
    """select_lists at the sizes that take the sieve, in one pass (exact and
    too small room) and in two, against the reference arithmetic."""
    from imaged11_amd import indexing
    assert batched.mfma_pays(K, N)
    ubi, gv = make(K, N, N)
    u, g = T(ubi, dev), T(gv, dev)
    thr = tol * tol
    n = batched.score_many(u, g, tol, exact=True).cpu().numpy()
    want = []
    for k in range(0, K, max(1, K // 5)):
        h = gv @ ubi[k].T
        d = ((h - np.rint(h)) ** 2).sum(1)
        edge = np.abs(d - thr) < 1e-12
        want.append((k, np.nonzero(d < thr)[0], edge.any()))
    for counts in (None, n, np.maximum(n // 2, 1), n + 5):
        idx, off = indexing.select_lists(u, g, thr, counts=counts)
        idx, off = idx.cpu().numpy(), off.cpu().numpy()
        assert np.array_equal(np.diff(off), n)
        for k, w, edge in want:
            got = idx[off[k]:off[k + 1]]
            assert np.all(np.diff(got) > 0)
            assert edge or np.array_equal(got, w)


# beyond the sieves' tolerances: the ball (tile edges, the accumulator's
# ranges, values that are not finite, distances at the tolerance)
@pytest.mark.parametrize("K,N", [(1, 1), (1, 5000), (31, 127), (33, 129), (65, 513), (2049, 700)])
@pytest.mark.parametrize("tol", [0.1001, 0.25, 0.499, 0.7499, 0.7501])
def test_ball_counts_at_tile_edges(dev, orc, K, N, tol):
    ubi, gv = make(K, N, K + N)
    for sign in (1, -1):
        got = batched.score_sieve(T(ubi, dev), T(gv, dev), sign * tol)
        assert np.array_equal(got.cpu().numpy(), orc.score_many(ubi, gv, tol))


@pytest.mark.parametrize("cell,gmax", [((10.0, 20.0), 1.6), ((20.0, 60.0), 1.6),
                                       ((200.0, 320.0), 1.6), ((300.0, 900.0), 1.6),
                                       ((900.0, 2000.0), 0.01), ((1e-4, 2e-4), 1e4),
                                       ((2e6, 5e6), 1e-6)])
def test_ball_over_the_ranges_of_the_accumulator(dev, orc, cell, gmax):
    ubi, gv = make(70, 3000, 5, cell=cell, gmax=gmax)
    for tol in (0.15, 0.3):
        got = batched.score_sieve(T(ubi, dev), T(gv, dev), tol)
        assert np.array_equal(got.cpu().numpy(), orc.score_many(ubi, gv, tol))


def test_ball_special_values(dev, orc):
    ubi, gv = make(40, 1000, 11)
    for i, v in enumerate([np.nan, np.inf, -np.inf, 1e300, 1e-310, 0.0]):
        gv[17 * i + 3, i % 3] = v
        gv[17 * i + 5] = v
        ubi[2 * i, i % 3, (i + 1) % 3] = v
        ubi[2 * i + 13] = v
    for u, g in ((ubi, gv), (ubi[:13:2], gv), (ubi[30:], gv[200:])):
        for tol in (0.25, 0.74):
            got = batched.score_sieve(T(u, dev), T(g, dev), tol)
            assert np.array_equal(got.cpu().numpy(), orc.score_many(u, g, tol))


def nonfinite_inputs():
    """Three tiles of grains and eight waves of peaks without a huge finite
    value, so that none of them leaves the matrix cores: in the first tile
    and its neighbour UBIs with one, two and three rows that are not finite
    (an entry, a row, entries in both rows), and peaks with one and three
    components that are not."""
    ubi, gv = make(96, 1024, 12)
    n = 0
    for v in (np.nan, np.inf, -np.inf):
        for rows in ((0,), (1,), (2,), (0, 1), (1, 2), (0, 2), (0, 1, 2)):
            ubi[2 * n, rows, n % 3] = v
            n += 1
        ubi[50 + n % 7, n % 3] = v  # a whole row
    for i, v in enumerate((np.nan, np.inf, -np.inf)):
        gv[40 * i + 3, i] = v
        gv[40 * i + 300] = v
    spans = np.abs(np.where(np.isfinite(ubi), ubi, 0.0)).sum(2).max()
    assert spans * np.abs(gv[np.isfinite(gv)]).max() < 60  # GS_SIEVE_SPAN
    return ubi, gv


@pytest.mark.parametrize("tol", [0.02, 0.1, 0.25, 0.501, 0.55, 0.6, 0.7, 0.709, 0.74])
def test_nonfinite_values_on_the_matrix_cores(dev, orc, tol):
    """A pair with a value that is not finite has a NaN drlv2: never counted,
    whichever rows it leaves finite."""
    ubi, gv = nonfinite_inputs()
    for scale in (1.0, 12.0):  # the narrow range and the wide one
        got = batched.score_sieve(T(ubi * scale, dev), T(gv, dev), tol).cpu().numpy()
        want = orc.score_many(ubi * scale, gv, tol)
        assert np.all(want[~np.isfinite(ubi).all((1, 2))] == 0) and want.sum() > 0
        assert np.array_equal(got, want)


@pytest.mark.parametrize("tol", [0.05, 0.25, 0.6, 0.74])
def test_huge_values_beside_nonfinite_ones(dev, orc, tol):
    """A huge finite entry in another row of a UBI that is not finite, and in
    tiles and waves of its own."""
    ubi, gv = nonfinite_inputs()
    ubi[0, 1, 1] = 1e300   # beside the NaN of row 0
    ubi[90, 2, 0] = -1e300
    gv[900, 1] = 1e300
    got = batched.score_sieve(T(ubi, dev), T(gv, dev), tol).cpu().numpy()
    assert np.array_equal(got, orc.score_many(ubi, gv, tol))


# tiles past the f16 ranges, tested in f32: spans from just beyond them to
# where f32 says nothing, factors up to the ends of f32 and past them
@pytest.mark.parametrize("cell,gmax", [((700.0, 1100.0), 1.6), ((3.0, 9.0), 40.0),
                                       ((0.3, 0.9), 90.0), ((9e3, 2.5e4), 1.6),
                                       ((3e4, 3e5), 1.6), ((1e28, 3e28), 1e-27),
                                       ((1e33, 3e33), 1e-32), ((1e-32, 3e-32), 1e33),
                                       ((1e-44, 3e-44), 1e45), ((1e40, 3e40), 1e-39)])
@pytest.mark.parametrize("K,N", [(33, 129), (64, 1000), (95, 2049)])
def test_tiles_in_f32(dev, orc, cell, gmax, K, N):
    ubi, gv = make(K, N, K, cell=cell, gmax=gmax)
    for tol in (0.0, 0.02, 0.1, 0.15, 0.45, 0.74):
        got = batched.score_sieve(T(ubi, dev), T(gv, dev), tol)
        want = orc.score_many(ubi, gv, tol)
        assert tol < 0.1 or want.sum() > 0
        assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("tol", [0.02, 0.1, 0.25, 0.6, 0.74])
def test_nonfinite_values_in_f32(dev, orc, tol):
    """The same values in tiles that are tested in f32, beside grains in
    range and grains whose every pair is settled."""
    ubi, gv = nonfinite_inputs()
    ubi[:32] *= 300.0  # past the f16 ranges
    ubi[32:64:5] *= 1e5  # and those of f32
    ubi[61, 1, 1], gv[900, 1] = 1e300, -1e300
    got = batched.score_sieve(T(ubi, dev), T(gv, dev), tol).cpu().numpy()
    want = orc.score_many(ubi, gv, tol)
    assert want[:32].sum() > 0 and want[64:].sum() > 0
    assert np.array_equal(got, want)


@pytest.mark.parametrize("cell,gmax", [((700.0, 1100.0), 1.6), ((0.3, 0.9), 90.0),
                                       ((3e4, 3e5), 1.6)])
def test_selected_lists_in_f32(dev, cell, gmax):
    from imaged11_amd import indexing
    K, N, tol = 700, 30001, 0.05
    ubi, gv = make(K, N, 2, cell=cell, gmax=gmax)
    u, g = T(ubi, dev), T(gv, dev)
    assert batched.mfma_pays(K, N)
    idx, off = indexing.select_lists(u, g, tol * tol)
    n = batched.score_many(u, g, tol, exact=True)
    assert np.array_equal(np.diff(off.cpu().numpy()), n.cpu().numpy())
    for k in range(0, K, 97):
        h = gv @ ubi[k].T
        d = ((h - np.rint(h)) ** 2).sum(1)
        got = idx[off[k]:off[k + 1]].cpu().numpy()
        scale = 1e-15 * np.abs(ubi[k]).sum() * np.abs(gv).max()  # of h in float64
        assert np.abs(d - tol * tol).min() < scale or np.array_equal(got, np.nonzero(d < tol * tol)[0])


@pytest.mark.parametrize("tol", [0.125, 0.3, 0.49])
def test_ball_pairs_on_the_tolerance(dev, orc, tol):
    """Distances that straddle tol by 1e-17 .. 1e-3, along one row, two and
    three: certain and settled pairs side by side in one quad."""
    a, rng = 4.0, np.random.default_rng(2)
    d = np.array([tol * (1 + s * 10.0 ** -e) for s in (-1, 1) for e in range(3, 17)])
    gv = []
    for axes in ((1, 0, 0), (0, -1, 0), (1, 1, 0), (1, -1, 1), (0, 2, 1)):
        v = np.array(axes, float)
        for h in rng.integers(-6, 7, (20, 3)):
            gv.append((h + d[:, None] * v / np.linalg.norm(v)) / a)
    gv = rng.permutation(np.concatenate(gv))
    ubi = np.eye(3)[None] * a * np.array([1.0, -1.0, 1.0])[:, None, None]
    got = batched.score_sieve(T(ubi, dev), T(gv, dev), tol).cpu().numpy()
    want = orc.score_many(ubi, gv, tol)
    assert 0 < want[0] < len(gv)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("K,N", [(15, 2200000), (16, 2000000), (321, 100001)])
def test_ball_dispatch(dev, K, N):
    """score_many's own choice against the FP64 kernel, on both sides of the
    rule; tol 0.74, 0.75 and 0.1 lie at its ends."""
    ubi, gv = make(K, N, 3)
    ubi, gv = T(ubi, dev), T(gv, dev)
    for tol in (0.1, 0.11, 0.25, 0.74, 0.75):
        assert torch.equal(batched.score_many(ubi, gv, tol),
                           batched.score_many(ubi, gv, tol, mode=_lib.SCORE_CERTIFIED))


# the kernels on the vector ALU: every call with labels of its own and every
# tol > 0.1, over the ends of their LDS chunks (512 and 1024 grains)
@pytest.mark.parametrize("K", [511, 512, 513, 1100])
@pytest.mark.parametrize("own,tol", [(True, 0.05), (False, 0.2)])
def test_scan_in_chunks_of_grains(dev, orc, K, own, tol):
    N = 3000
    ubi, trans, xl, so, co, w, rng = scan_inputs(K, N, K)
    gl = rng.permutation(K + 50)[:K].astype(np.int32) if own else np.arange(K, dtype=np.int32)
    d0, l0 = rng.uniform(0, 0.1, N), rng.integers(-2, K + 50, N).astype(np.int32)
    d, lab = d0.copy(), l0.copy()
    want = orc.gv_assign_many(xl, so, co, np.eye(3), w, ubi, trans, gl, tol, d, lab)
    dd, ll = T(d0, dev), T(l0, dev, torch.int32)
    got = batched.gv_assign_many(T(xl, dev), T(so, dev), T(co, dev), w, T(ubi, dev), T(trans, dev),
                                 tol, dd, ll, grain_labels=T(gl, dev, torch.int32) if own else None,
                                 mat=np.eye(3))
    assert want.sum() > 0 and np.array_equal(got.cpu().numpy(), want)
    assert np.array_equal(ll.cpu().numpy(), lab)
    assert np.array_equal(dd.cpu().numpy().view(np.int64), d.view(np.int64))


@pytest.mark.parametrize("K", [1023, 1024, 1025, 2100])
@pytest.mark.parametrize("own,tol", [(True, 0.05), (False, 0.2)])
def test_assignment_in_chunks_of_grains(dev, orc, K, own, tol):
    N = 2500
    ubi, gv = make(K, N, K)
    rng = np.random.default_rng(K)
    gl = rng.permutation(K + 50)[:K].astype(np.int32) if own else np.arange(K, dtype=np.int32)
    d0, l0 = rng.uniform(0, 0.1, N), rng.integers(-2, K + 50, N).astype(np.int32)
    d, lab = d0.copy(), l0.copy()
    want = orc.assign_many(ubi, gl, gv, tol, d, lab)
    dd, ll = T(d0, dev), T(l0, dev, torch.int32)
    got = batched.assign_many(T(ubi, dev), T(gv, dev), tol, dd, ll,
                              grain_labels=T(gl, dev, torch.int32) if own else None)
    assert want.sum() > 0 and np.array_equal(got.cpu().numpy(), want)
    assert np.array_equal(ll.cpu().numpy(), lab)
    assert np.array_equal(dd.cpu().numpy().view(np.int64), d.view(np.int64))
