"""P + P^T with rows longer than a wave sorts: the values against the FP64 oracle, and their share of the time."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _graph(n, rows, cols, rng):
    pair = np.unique(rows.astype(np.int64) * n + cols)
    rows, cols = pair // n, pair % n
    rows, cols = rows[rows != cols], cols[rows != cols]
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, rows + 1, 1)
    return np.cumsum(rp), cols.astype(np.int32), rng.uniform(0.1, 1.0, rows.size).astype(np.float32)


def _hubs(n, hubs, degree, rng, k=3):
    """Every vertex has k neighbours, and the hubs `degree` more that point at them and that they point at."""
    i = np.arange(n)
    rows, cols = [np.repeat(i, k)], [(i[:, None] + 1 + 5 * np.arange(k)[None]).ravel() % n]
    for h in hubs:
        v = rng.permutation(n)[:degree]
        rows += [v, np.full(degree // 2, h)]
        cols += [np.full(degree, h), v[: degree // 2]]
    return _graph(n, np.concatenate(rows), np.concatenate(cols), rng)


def _check(sg, O, n, rp, col, val):
    with sg.Context(sg.tsneparams(reorder=0)) as ctx:
        ctx.upload_P(sg.CSR(n, rp, col, val), symmetrize=True)
        P = ctx.get_P()
    S = O.symmetrize(O.CSR(n, rp.astype(np.int64), col, val.astype(np.float64)))
    assert np.array_equal(P.rowptr, S.rowptr) and np.array_equal(P.col, S.col)
    # FP64 sums in another order, rounded once to FP32
    assert np.all(np.abs(P.val - S.val) <= 2.0**-24 * S.val * (1 + 1e-6))


# hubs whose columns end in, fill and exceed ranges of 8192; a hub whose columns
# need more than one bitmap of 524,288 below them; rows on the first and last vertex
@pytest.mark.parametrize("n,hubs,degree", [(8192, (0, 8191), 8000), (8193, (8192,), 8190), (16385, (1, 7, 16384), 12000),
                                           (40000, (39999, 0), 39000), (540000, (3, 539999), 530000)])
def test_symmetrize_hubs(sg, O, n, hubs, degree):
    rng = np.random.default_rng(n)
    _check(sg, O, n, *_hubs(n, hubs, degree, rng))


# every row longer than a wave sorts, on both sides of a work-group's limit
@pytest.mark.parametrize("n,k", [(1500, 900), (3001, 1100), (9000, 5000)])
def test_symmetrize_every_row_long(sg, O, n, k):
    rng = np.random.default_rng(n + k)
    cols = np.concatenate([rng.permutation(n)[:k] for _ in range(n)])
    _check(sg, O, n, *_graph(n, np.repeat(np.arange(n), k), cols, rng))


# entries of a hub given three times, and one of value zero
def test_symmetrize_hub_duplicates(sg, O):
    n, rng = 30000, np.random.default_rng(4)
    rp, col, val = _hubs(n, (100,), 20000, rng)
    rows = np.repeat(np.arange(n), np.diff(rp))
    val[np.flatnonzero(col == 100)[::7]] = 0.0
    rows, col, val = np.repeat(rows, 3), np.repeat(col, 3), np.repeat(val, 3)
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, rows + 1, 1)
    _check(sg, O, n, np.cumsum(rp), col, val)


# eight hubs of 100,000 entries among 4 M others cost about what their entries do
# (a sort per row in memory by one work-group took 20 times the whole)
def test_symmetrize_hubs_cost_their_entries(sg):
    n, rng = 200000, np.random.default_rng(9)
    with sg.Batch(sg.tsneparams(d=2), 2, n + 64, 12_000_000) as B:

        def ms(hubs):
            rp, col, val = _hubs(n, hubs, 100000, rng, k=20)
            P, y0 = sg.CSR(n, rp, col, val), rng.standard_normal((n, 2)).astype(np.float32)
            best = 1e9
            for _ in range(5):
                t = time.perf_counter()
                j = B.add(P, y_in=y0, max_iter=2)
                B.sync()
                best = min(best, time.perf_counter() - t)
                B.remove(j)
                B.sync()
            return best

        assert ms(range(0, 8000, 1000)) < 4 * ms(())
