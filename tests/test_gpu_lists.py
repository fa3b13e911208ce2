"""Peak lists from labels and the visiting order against numpy."""
import numpy as np
import pytest
import torch

from imaged11_amd import _lib, batched

pytestmark = pytest.mark.gpu


def reference(lab, K):
    idx = [np.nonzero(lab == g)[0] for g in range(K)]
    off = np.concatenate([[0], np.cumsum([len(i) for i in idx])]).astype(np.int64)
    return (np.concatenate(idx) if K else np.zeros(0, int), off,
            np.repeat(np.arange(K), np.diff(off)))


@pytest.mark.parametrize("n,K", [(0, 5), (7, 0), (1, 1), (64, 3), (1000, 1), (5000, 70),
                                 (100001, 777), (300000, 5000), (40000, 2100)])
def test_lists(dev, n, K):
    rng = np.random.default_rng(n + K)
    # heavy and empty lists, labels outside [0, K)
    lab = np.minimum(rng.integers(-2, K + 3, n), rng.integers(-1, K + 2, n)).astype(np.int32)
    lab[lab == 2] = 1
    want = reference(lab, K)
    for t in (torch.as_tensor(lab, device=dev), torch.as_tensor(lab, device=dev).long()):
        got = batched.lists_from_labels(t, K)
        assert [g.dtype for g in got] == [torch.int32, torch.int64, torch.int32]
        for g, w in zip(got, want):
            assert np.array_equal(g.cpu().numpy(), w)
        assert np.array_equal(batched.label_counts(t, K).cpu().numpy(), np.diff(want[1]))


@pytest.mark.parametrize("longest", [_lib.LIST_SORT_MAX - 1, _lib.LIST_SORT_MAX,
                                     _lib.LIST_SORT_MAX + 1])
def test_the_longest_list(dev, longest):
    rng = np.random.default_rng(3)
    lab = rng.permutation(np.concatenate([np.full(longest, 4), rng.integers(-1, 4, 3000)]))
    lab = lab.astype(np.int32)
    for g, w in zip(batched.lists_from_labels(torch.as_tensor(lab, device=dev), 6),
                    reference(lab, 6)):
        assert np.array_equal(g.cpu().numpy(), w)


@pytest.mark.parametrize("K", [1, 63, 64, 65, 1000, _lib.ORDER_MAX, _lib.ORDER_MAX + 1])
def test_order(dev, K):
    rng = np.random.default_rng(K)
    length = rng.integers(0, 40, K)
    length[::5] = rng.integers(0, 1 << 33, length[::5].shape)
    off = np.concatenate([[0], np.cumsum(length)])
    got = batched.list_order(torch.as_tensor(off, device=dev))
    assert got.dtype == torch.int32
    assert np.array_equal(got.cpu().numpy(), np.argsort(-length, kind="stable"))


@pytest.mark.parametrize("K", [_lib.LIST_GRAINS_MAX, _lib.LIST_GRAINS_MAX + 1])
def test_lists_of_many_grains(dev, K):
    assert batched.list_kernels_pay(K) == (K <= _lib.LIST_GRAINS_MAX)
    rng = np.random.default_rng(K)
    lab = rng.integers(-1, K, 3000).astype(np.int32)
    lab[-1] = K - 1
    idx, off, owner = (g.cpu().numpy() for g in batched.lists_from_labels(
        torch.as_tensor(lab, device=dev), K))
    order = np.argsort(np.where(lab < 0, K, lab), kind="stable")[:(lab >= 0).sum()]
    assert np.array_equal(idx, order) and np.array_equal(owner, lab[order])
    assert np.array_equal(off, np.searchsorted(lab[order], np.arange(K + 1)))


def test_few_of_many_labels_stay_with_the_kernels(dev, monkeypatch):
    """Short lists among a great many peaks of no grain."""
    n, K = 8 * _lib.LIST_SORT_MAX, 2
    lab = np.full(n, -1, np.int32)
    lab[5::1000] = np.arange(len(lab[5::1000])) % K
    t = torch.as_tensor(lab, device=dev)
    monkeypatch.setattr(torch, "nonzero", None)  # torch's route
    got = batched.lists_from_labels(t, K)
    for g, w in zip(got, reference(lab, K)):
        assert np.array_equal(g.cpu().numpy(), w)
