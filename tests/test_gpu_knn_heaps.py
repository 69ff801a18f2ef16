"""Exact kNN of many points, whose rows come from heaps instead of blocks of distances."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _points(n, dim, seed):
    rng = np.random.default_rng(seed)
    c = rng.normal(0, 4, (10, dim))
    return (c[rng.integers(0, 10, n)] + rng.standard_normal((n, dim))).astype(np.float32)


# the last work-group's 64 queries and the last 32 references are cut short, the
# dimensions of a round of 16 are; the smallest search of the heaps; k above 256
@pytest.mark.parametrize("n,dim,k", [(16385, 1, 1), (40003, 17, 10), (60007, 5, 90), (100_000, 130, 3), (120_001, 3, 300)])
def test_knn_exact_by_heaps(sg, O, n, dim, k):
    X = _points(n, dim, n)
    X[5] = X[n - 1]  # the nearest point of each other, at distance zero
    X[::997, 0] = X[3, 0]
    I, D, fb = sg.knn(X, k, sg.KNN_EXACT_FP64)
    assert fb == -1
    rows = np.unique(np.r_[0:70, 5, n // 2, n - 70:n].astype(np.int32))
    Io, Do = O.knn_rows(X, k, rows)
    assert np.array_equal(I[rows], Io) and np.array_equal(D[rows], Do)


def test_knn_exact_by_heaps_points_without_neighbours(sg):
    n, k = 20_011, 5
    X = _points(n, 2, 1)
    X[7] = np.nan
    X[n - 1] = np.inf  # as far from every point as any
    I, D, _ = sg.knn(X, k, sg.KNN_EXACT_FP64)
    assert I[7, 0] == 7 and (I[7, 1:] == np.iinfo(np.int32).max).all() and np.isposinf(D[7, 1:]).all()
    assert np.array_equal(I[n - 1], [n - 1, 0, 1, 2, 3, 4]) and np.isposinf(D[n - 1, 1:]).all()
    ok = np.delete(np.arange(n), [7, n - 1])
    assert np.isfinite(D[ok]).all() and not np.isin(I[ok], [7, n - 1]).any()


# rows the certificate leaves, enough of them for the heaps: equal points, whose
# neighbours are the equal points of lowest index
def test_knn_uncertified_rows_by_heaps(sg):
    n, dim, k, m = 60_000, 5, 10, 12_001
    X = _points(n, dim, 2)
    same = np.sort(np.random.default_rng(3).permutation(n)[:m])
    X[same] = X[same[0]]
    I, D, fb = sg.knn(X, k, sg.KNN_FILTERED)
    assert fb >= m
    first = same[:k + 1]
    want = np.array([np.r_[q, first[first != q][:k]] for q in same])
    assert np.array_equal(I[same], want) and not D[same].any()


# four times the points are sixteen times the pairs; half as much again for what
# does not grow evenly.  With every distance stored and selected in blocks of 512 MB
# 60,000 points took 35.6 ms and 200,000, eleven times the pairs, 957; heaps 8.2 and 78
def test_knn_exact_cost_per_pair(sg):
    def ms(n):
        X = _points(n, 5, 4)
        best = 1e9
        for _ in range(3):
            t = time.perf_counter()
            sg.knn(X, 10, sg.KNN_EXACT_FP64)
            best = min(best, time.perf_counter() - t)
        return best

    small, large = ms(60_000), ms(240_000)
    assert large <= 24 * small, (small, large)
