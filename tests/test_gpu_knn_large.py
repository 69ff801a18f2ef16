"""Uncertified rows of a search over so many points that a block of exact distances is 128 of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_knn_exact_rows_of_a_large_search(sg):
    n, dim, k, m = 530_000, 8, 20, 300
    rng = np.random.default_rng(6)
    c = rng.normal(0, 4, (20, dim))
    X = (c[rng.integers(0, 20, n)] + rng.standard_normal((n, dim))).astype(np.float32)
    same = np.sort(rng.permutation(n)[:m])  # more ties at distance zero than the candidate lists hold
    X[same] = X[same[0]]
    I, D, fb = sg.knn(X, k, sg.KNN_FILTERED)
    assert fb >= m
    for q in same:
        want = same[same != q][:k]  # ties by index
        assert I[q, 0] == q and np.array_equal(I[q, 1:], want) and not D[q].any()
