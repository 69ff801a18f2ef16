"""kNN kernels at the edges of their tiles: rows bit for bit against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sg():
    import sgtsne_amd

    return sgtsne_amd


@pytest.fixture(scope="module")
def O():
    from oracle import oracle

    return oracle


def _points(n, dim, seed):
    rng = np.random.default_rng(seed)
    centres = rng.normal(0, 4, size=(6, dim))
    return (centres[rng.integers(0, 6, n)] + rng.standard_normal((n, dim))).astype(np.float32)


# one point beyond / at / under the 128 x 128 tiles, dimensions around the 16
# staged at a time, k around the two selection widths
@pytest.mark.parametrize("n,dim,k", [(2, 1, 1), (127, 16, 126), (128, 17, 40), (129, 1, 3), (257, 15, 256), (300, 130, 257),
                                     (700, 784, 90), (2100, 5, 2048), (1000, 33, 600)])
def test_knn_exact_tiles(sg, O, n, dim, k):
    X = _points(n, dim, n + dim)
    I, D, fb = sg.knn(X, k, sg.KNN_EXACT_FP64)
    Io, Do = O.knn_exact(X, k)
    assert fb == -1 and np.array_equal(I, Io) and np.array_equal(D, Do)


@pytest.mark.parametrize("n,distinct,k", [(3000, 2, 90), (3000, 1, 300), (5000, 7, 20)])
def test_knn_exact_wide_ties(sg, O, n, distinct, k):
    # far more keys tie at the k-th smallest than the selection sorts
    X = np.repeat((np.arange(n) % distinct).astype(np.float32)[:, None], 3, axis=1)
    I, D, _ = sg.knn(X, k, sg.KNN_EXACT_FP64)
    Io, Do = O.knn_exact(X, k)
    assert np.array_equal(I, Io) and np.array_equal(D, Do)


def test_knn_exact_infinite_points(sg):
    # a pair with one infinite point is infinitely far (taken by index after
    # every finite one), a pair of them has no distance (NaN) and is no neighbour
    X = _points(200, 4, 8)
    X[[3, 50, 199], 1] = np.inf
    I, D, _ = sg.knn(X, 198, sg.KNN_EXACT_FP64)
    far = [3, 50, 199]
    assert I[0, -2:].tolist() == [3, 50] and np.isinf(D[0, -2:]).all() and np.isfinite(D[0, :-2]).all()
    near = [i for i in range(200) if i not in far]
    assert I[3, 1:198].tolist() == near and np.isinf(D[3, 1:]).all() and I[3, 198] == np.iinfo(np.int32).max


# query blocks and reference tiles one point short / full / one over, every
# step count of the filter's template, lists at their largest (k + 16 = 128)
@pytest.mark.parametrize("n,dim,k", [(64, 3, 40), (65, 16, 30), (129, 17, 112), (193, 31, 90), (1000, 48, 112), (1025, 49, 16),
                                     (2048, 64, 90), (3001, 96, 45), (2500, 100, 1)])
def test_knn_filtered_lists(sg, O, n, dim, k):
    X = _points(n, dim, 3 * n + dim)
    I, D, fb = sg.knn(X, k, sg.KNN_FILTERED)
    Io, Do = O.knn_exact(X, k)
    assert fb >= 0 and np.array_equal(I, Io) and np.array_equal(D, Do)


@pytest.mark.parametrize("step", [1.0, -1.0])
def test_knn_filtered_every_reference_enters(sg, O, step):
    # points on a line, ever farther from (or nearer to) the first ones: in one
    # direction every reference beats the list's threshold as it is visited
    n = 4000
    X = np.zeros((n, 4), np.float32)
    X[:, 0] = step * np.arange(n, dtype=np.float32) ** 1.5
    I, D, fb = sg.knn(X, 90, sg.KNN_FILTERED)
    Io, Do = O.knn_exact(X, 90)
    assert np.array_equal(I, Io) and np.array_equal(D, Do)


def test_knn_filtered_wide_blocks(sg):
    # the 32-query work-groups of very large jobs, on rows sampled from one
    X = _points(530_000, 8, 4)
    I, D, fb = sg.knn(X, 20, sg.KNN_FILTERED)
    rows = np.arange(0, X.shape[0], 1877)
    Xd = X.astype(np.float64)
    for q in rows:
        d2 = ((Xd - Xd[q]) ** 2).sum(1)
        d2[q] = np.inf
        near = np.sort(np.partition(d2, 19)[:20])
        assert I[q, 0] == q and np.allclose(D[q, 1:], near, rtol=1e-12) and np.allclose(d2[I[q, 1:]], near, rtol=1e-12)


# candidate lists of 65..256 entries re-ranked by one wave, two and four to a
# lane, rows staged 16 dimensions at a time with a remainder
@pytest.mark.parametrize("n,dim,k", [(66, 18, 64), (400, 20, 112), (401, 17, 113), (500, 18, 200), (900, 20, 240), (250, 64, 240)])
def test_knn_filtered_rerank_widths(sg, O, n, dim, k):
    X = _points(n, dim, 5 * n + dim)
    I, D, fb = sg.knn(X, k, sg.KNN_FILTERED)
    Io, Do = O.knn_exact(X, k)
    assert fb >= 0 and np.array_equal(I, Io) and np.array_equal(D, Do)


# both sides of the points up to which the filter gives a query block 16 waves
# (where the dimensions leave the registers) and eight
@pytest.mark.parametrize("n,dim", [(4096, 64), (4096, 65), (4097, 64), (32768, 12), (32769, 12)])
def test_knn_filtered_wave_counts(sg, n, dim):
    X = _points(n, dim, n)
    I, D, fb = sg.knn(X, 30, sg.KNN_FILTERED)
    Ie, De, _ = sg.knn(X, 30, sg.KNN_EXACT_FP64)
    assert fb >= 0 and np.array_equal(I, Ie) and np.array_equal(D, De)
