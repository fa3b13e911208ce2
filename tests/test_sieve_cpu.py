"""The error bound of the matrix-core sieve, in numpy: h from f16 pieces,
products exact, f32 accumulation that rounds or truncates at every step."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from imaged11_amd import batched, indexing


def split16(v):
    hi = np.float16(np.float32(v))
    return hi, np.float16(np.float32(v - hi.astype(np.float64)))


def accumulate(prods, start, mode, rng):
    """Sum of the k slots in a random order, every addition rounded to f32
    to nearest or towards zero."""
    acc = np.full(prods.shape[0], np.float32(start))
    for k in rng.permutation(prods.shape[1]):
        s = acc.astype(np.float64) + prods[:, k]
        f = s.astype(np.float32)
        if mode == "truncate":
            over = np.abs(f.astype(np.float64)) > np.abs(s)
            f = np.where(over, np.nextafter(f, np.float32(0)), f)
        acc = f
    return acc


@pytest.mark.parametrize("mode", ["nearest", "truncate"])
@pytest.mark.parametrize("span,start,err", [(60.0, 1.5 * 2.0 ** 23, 2.0 ** -11),
                                            (1000.0, 1.5 * 2.0 ** 27, 2.0 ** -7)])
def test_sieve_error_bound(mode, span, start, err):
    rng = np.random.default_rng(1)
    worst = 0.0
    for scale in (1e-3, 0.3, 4.0, 60.0, 800.0):
        n = 20000
        u = rng.uniform(-1, 1, (n, 3)) * scale
        gmax = min(29.9, span / np.abs(u).sum(1).max())
        g = rng.uniform(-1, 1, (n, 3)) * gmax
        g[::7] = np.sign(u[::7]) * gmax  # the largest sums
        uh, ul = split16(u * 64.0)
        gh, gl = split16(g * 1024.0)
        f = lambda a: a.astype(np.float64)
        prods = np.concatenate([f(gh) * f(uh), f(gl) * f(uh), f(gh) * f(ul)], 1)
        acc = accumulate(prods, start, mode, rng)
        assert np.all((acc >= start * 2 / 3) & (acc < start * 4 / 3))  # one binade
        h = (acc.astype(np.float64) - start) / 65536.0
        exact = (u.astype(np.longdouble) * g.astype(np.longdouble)).sum(1)
        worst = max(worst, float(np.abs(h - exact).max()))
    assert worst < err
    assert worst > err / 200  # the test reaches the range the bound is for


@pytest.mark.parametrize("ratio", [1e-4, 2e-3, 0.03, 0.1, 0.2])
def test_position_expansion_error_bound(ratio):
    """u.G for a grain at t against the sieve's terms: G0 and the products p q
    with p and q rounded to f16, over t/|a| up to the largest sieved."""
    rng = np.random.default_rng(2)
    n, ds, amin = 20000, 5.0, 150000.0
    a = rng.normal(size=(n, 3))
    a *= (amin * rng.uniform(1.0, 1.3, n) / np.linalg.norm(a, axis=1))[:, None]
    t = rng.normal(size=(n, 3))
    t *= (ratio * amin * rng.uniform(0.0, 1.0, n) / np.linalg.norm(t, axis=1))[:, None]
    t[::5] = np.cross(a[::5], [0.3, -0.5, 0.8])  # across the beam: the largest remainder
    t[::5] *= ratio * amin / np.linalg.norm(t[::5], axis=1)[:, None]
    u = rng.uniform(-9, 9, (n, 3))
    e = a - t
    exact = (u * (ds * e / np.linalg.norm(e, axis=1)[:, None])).sum(1)
    r = np.linalg.norm(a, axis=1)
    nn = a / r[:, None]
    i, j = np.array([0, 1, 2, 0, 0, 1]), np.array([0, 1, 2, 1, 2, 2])
    y = 4 - int(np.frexp(np.abs(t).max())[1])
    p = (ds / r)[:, None] * nn[:, i] * nn[:, j]
    q = u[:, i] * t[:, j] + u[:, j] * t[:, i]
    q[:, :3] = u * t - (u * t).sum(1)[:, None]
    p16 = np.float16(np.float32(p * 2.0 ** (16 - y))).astype(float)
    q16 = np.float16(np.float32(q * 2.0 ** y)).astype(float)
    assert p16.max() < 8192 and np.isfinite(q16).all()
    approx = (u * (ds * nn)).sum(1) + (p16 * q16).sum(1) / 65536.0
    L, A1, T = np.abs(q).sum(1), np.abs(u).sum(1), np.linalg.norm(t, axis=1)
    bound = 1.01 * 2.0 ** -10 * ds / amin * L + 0.5775 * A1 * ds * (T / (amin - T)) ** 2
    assert np.all(np.abs(approx - exact) <= bound + 1e-12)


@pytest.mark.parametrize("window", [8.0, 32.0, 64.0, 160.0])
@pytest.mark.parametrize("ratio", [1e-4, 0.01, 0.06])
def test_position_expansion_over_the_exponents(window, ratio):
    """The same with 2^y anywhere between 8 and 160 ds/|a|, numbers below the
    normal f16 range flushed to zero: p within 8192, sum |q| within 32768
    wherever the radius stays below 0.2, and the flushed terms within their
    2^-30 (32768 + 2 8192)."""
    rng = np.random.default_rng(5)
    n, ds, amin = 20000, 5.0, 150000.0
    a = rng.normal(size=(n, 3))
    a *= (amin * rng.uniform(1.0, 1.3, n) / np.linalg.norm(a, axis=1))[:, None]
    t = rng.normal(size=(n, 3)) * 10.0 ** rng.uniform(-9, 0, (n, 3))
    t *= (ratio * amin * rng.uniform(0.0, 1.0, n) / np.linalg.norm(t, axis=1))[:, None]
    u = rng.uniform(-9, 9, (n, 3)) * 10.0 ** rng.uniform(-6, 0, (n, 3))
    y = int(np.floor(np.log2(window * ds / amin)))
    if 2.0 ** y < 8 * ds / amin:
        y += 1
    r = np.linalg.norm(a, axis=1)
    nn = a / r[:, None]
    i, j = np.array([0, 1, 2, 0, 0, 1]), np.array([0, 1, 2, 1, 2, 2])
    p = (ds / r)[:, None] * nn[:, i] * nn[:, j]
    q = u[:, i] * t[:, j] + u[:, j] * t[:, i]
    q[:, :3] = u * t - (u * t).sum(1)[:, None]
    L = np.abs(q).sum(1)
    sieved = 1.01 * 2.0 ** -10 * ds / amin * L < 0.2
    f = lambda v: np.float16(np.float32(v)).astype(float)
    p16, q16 = f(p * 2.0 ** (16 - y)), f(q * 2.0 ** y)
    assert np.abs(p16).max() <= 8192 and (L * 2.0 ** y)[sieved].max() <= 32768
    near = (p16 * q16).sum(1) / 65536.0
    flush = lambda v: np.where(np.abs(v) < 2.0 ** -14, 0.0, v)
    gone = np.abs((flush(p16) * flush(q16)).sum(1) / 65536.0 - near)
    assert gone[sieved].max() <= 2.0 ** -30 * (32768 + 2 * 8192)
    err = np.abs(near - (p * q).sum(1)) - 1.01 * 2.0 ** -10 * ds / amin * L
    assert err[sieved].max() <= 2.0 ** -30 * (32768 + 2 * 8192)


def fma32(a, b, c):
    """f32 FMA: the product of two f32 is exact in f64 (the sum's rounding there
    is 2^-29 of the rounding to f32)."""
    return (a.astype(np.float64) * b.astype(np.float64) + c).astype(np.float32)


@pytest.mark.parametrize("span", [1e-3, 1.0, 60.0, 1000.0, 16384.0, 65536.0])
def test_f32_tile_error_bound(span):
    """h + r of gs_cube32 within 2^-21 A + 10^-6, and drlv2 of gs_drlv2_32
    within the bounds gs_units32 draws around it."""
    rng = np.random.default_rng(3)
    n, worst = 200000, 0.0
    u = rng.uniform(-1, 1, (n, 3, 3))
    g = rng.uniform(-1, 1, (n, 3))
    g[::3] = np.sign(u[::3, 0]) * np.abs(g[::3]).max(1)[:, None]  # the largest sums
    u *= span / (np.abs(u).sum(2).max(1) * np.abs(g).max(1))[:, None, None]
    A = np.abs(u).sum(2).max(1) * np.abs(g).max(1)
    err = 2.0 ** -21 * A + 1e-6
    u32, g32 = u.astype(np.float32), g.astype(np.float32)
    f, d2 = [], []
    for row in range(3):
        exact = (u[:, row].astype(np.longdouble) * g.astype(np.longdouble)).sum(1)
        for start in (0.0501, 0.5):
            h = np.full(n, start, np.float32)
            for j in range(3):
                h = fma32(u32[:, row, j], g32[:, j], h.astype(np.float64))
            worst = max(worst, float((np.abs(h - (exact + np.float32(start))) / err).max()))
        f.append(h - np.floor(h))
        d2.append((exact - np.rint(exact)) ** 2)
    assert 0.05 < worst < 0.99
    t = fma32(f[0], f[0], -f[0].astype(np.float64))
    for k in (1, 2):
        t = fma32(f[k], f[k], t.astype(np.float64)) - f[k]
    root = np.sqrt(sum(d2).astype(float))
    d = 1.7320509 * err
    assert np.all(t >= np.maximum(root - d, 0) ** 2 - 0.750002)
    assert np.all(t <= (root + d) ** 2 - 0.749998)


@pytest.mark.parametrize("ratio", [1e-3, 0.05, 0.3, 0.5])
@pytest.mark.parametrize("cell", [3.0, 300.0, 12000.0])
def test_f32_position_error_bound(ratio, cell):
    """u.G of the assignment's f32 tiles, |t| up to half of |a|, with the
    inverse square root off by its 2 v either way: within 2^-19 A1 ds."""
    rng = np.random.default_rng(4)
    n, ds, amin = 100000, 5.0, 8000.0
    a = rng.normal(size=(n, 3))
    a *= (amin * rng.uniform(1.0, 3.0, n) / np.linalg.norm(a, axis=1))[:, None]
    t = rng.normal(size=(n, 3))
    t *= (ratio * amin * rng.uniform(0.0, 1.0, n) / np.linalg.norm(t, axis=1))[:, None]
    t[::3] = a[::3] * (ratio * amin / np.linalg.norm(a[::3], axis=1))[:, None]  # towards it
    c = rng.normal(size=(n, 3))
    c *= ds / np.linalg.norm(c, axis=1)[:, None]
    u = rng.uniform(-cell, cell, (n, 3))
    e = (a - t).astype(np.longdouble)
    G = ds * e / np.sqrt((e * e).sum(1))[:, None] - c
    exact = (u * G).sum(1)
    f = np.float32
    e32 = a.astype(f) - t.astype(f)
    n2 = e32[:, 0] * e32[:, 0]
    for j in (1, 2):
        n2 = fma32(e32[:, j], e32[:, j], n2.astype(np.float64))
    for off in (-1.0, 0.0, 1.0):
        rsq = (1.0 / np.sqrt(n2.astype(np.float64)) * (1.0 + off * 2.0 ** -23)).astype(f)
        inv = f(ds) * rsq
        h = np.full(n, f(0.0501))
        for j in range(3):
            g = fma32(e32[:, j], inv, -c[:, j].astype(f).astype(np.float64))
            h = fma32(u[:, j].astype(f), g, h.astype(np.float64))
        err = np.abs(h - f(0.0501) - exact) / (2.0 ** -19 * np.abs(u).sum(1) * ds + 1e-6)
        assert 0.02 < err.max() < 0.99


@pytest.mark.parametrize("err", [2.0 ** -11, 2.0 ** -7])
def test_dead_pairs_lie_beyond_the_ball(err):
    """A pair held at 1/2 in all three rows has S = 3/4, beyond lo + width at
    every tolerance the ball takes; held there in one row or two it would
    be certain from tol 1/2, sqrt(1/2) on, so the three go together."""
    def units(tol):
        e = 1.7320508075688774 * err + 1e-9
        lo = int(max((max(tol - e, 0.0) * 65536.0) ** 2 - 1.0, 0.0))
        return lo, int(((tol + e) * 65536.0) ** 2 + 2.0)

    for tol in np.linspace(0.1, 0.75, 131):
        lo, hi = units(tol)
        assert hi < 3 << 30
        for dead in (1, 2):  # the live rows at an integer
            if tol > np.sqrt(dead / 4.0) + 2 * np.sqrt(3.0) * err:
                assert dead << 30 < lo


def test_dispatch_stays_within_the_limits_of_the_kernels():
    """The queue entries of the assignment hold 24 bits of grain; the score's
    workspace is larger than the UBIs."""
    for K, assign, score in ((1 << 24, True, True), ((1 << 24) + 1, False, True),
                             (1 << 28, False, True), ((1 << 28) + 1, False, False),
                             ((1 << 31) - 1, False, False), (7, False, False)):
        assert batched.assign_mfma_pays(K, 10 ** 7, 0.05) == assign
        assert batched.mfma_pays(K, 10 ** 7) == score
        assert batched.score_mfma_pays(K, 10 ** 7, 0.05) == score
        assert batched.ball_pays(K, 10 ** 7, 0.3) == score


def test_few_grains_with_many_peaks_stay_with_the_vector_kernel():
    for K, N, pays in ((15, 100, False), (16, 300000, True), (19, 300001, False), (20, 10 ** 7, True)):
        assert batched.assign_mfma_pays(K, N, 0.05) == pays
        assert not batched.assign_mfma_pays(K, N, 0.11)


@pytest.mark.parametrize("K,pairs,narrow,wide", [
    (1, 10 ** 9, False, False), (15, 10 ** 8, False, False), (16, 16 * 10 ** 6, True, True),
    (16, 15999984, False, False), (32, 16 * 10 ** 6, True, True), (33, 23 * 10 ** 6, False, False),
    (33, 24 * 10 ** 6, True, True), (40, 64 * 10 ** 6, False, False), (40, 96 * 10 ** 6, True, True),
    (64, 24 * 10 ** 6, True, True), (72, 95 * 10 ** 6, False, False),
    (88, 96 * 10 ** 6, True, True), (96, 32 * 10 ** 6, False, True),
    (100, 48 * 10 ** 6, True, True), (256, 31 * 10 ** 6, False, False),
    (256, 48 * 10 ** 6, True, True), (257, 17 * 10 ** 6, False, False),
    (1000, 18 * 10 ** 6, True, True), (12000, 15 * 10 ** 6, False, False)])
def test_the_score_takes_the_matrix_cores_where_they_were_measured_faster(K, pairs, narrow, wide):
    """Both sides of every line of the rule."""
    N = -(-pairs // K)
    for sign in (1, -1):
        assert batched.score_mfma_pays(K, N, sign * 0.02) == narrow
        assert batched.score_mfma_pays(K, N, sign * 0.05) == wide


@pytest.mark.parametrize("index,current,ok", [(0, 0, True), (1, 0, False), (0, 1, False)])
def test_labels_of_another_device_stay_with_torch(monkeypatch, index, current, ok):
    """The list kernels launch on the current device's stream."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: current)
    labels = SimpleNamespace(is_cuda=True, device=torch.device("cuda", index), dtype=torch.int32,
                             dim=lambda: 1, is_contiguous=lambda: True, numel=lambda: 5)
    assert batched._int32_labels(labels) == ok
    assert not batched._int32_labels(torch.zeros(5, dtype=torch.int32))


@pytest.mark.parametrize("K,N,thr,pays", [(8, 2000000, 0.01, True), (8, 2000000, 0.1 ** 2, False),
                                          (16, 1000000, 0.1 ** 2, True), (16, 999999, 0.01, False),
                                          (1000, 16000, 0.0101, False), (7, 10 ** 8, 0.01, False)])
def test_selections_behind_the_sieve(K, N, thr, pays):
    assert indexing.sieve_pays(K, N, thr) == pays
