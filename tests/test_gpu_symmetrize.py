"""P + P^T at the edges of its row sizes, against the FP64 oracle."""
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


def _csr(n, rows, cols, rng):
    order = np.lexsort((rng.random(rows.size), rows))  # columns of a row in any order
    rows, cols = rows[order], cols[order]
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, rows + 1, 1)
    return np.cumsum(rp), cols.astype(np.int32), rng.uniform(0.1, 1.0, rows.size).astype(np.float32)


# hub: every vertex points at vertex 0, whose merged row has hub + 1 entries (with
# its own one): a wave's longest, one more, the LDS limit, beyond it, memory
@pytest.mark.parametrize("n,hub", [(5, 4), (1100, 1023), (1100, 1024), (8300, 8191), (8300, 8192), (20001, 20000)])
def test_symmetrize_hub(sg, O, n, hub):
    rng = np.random.default_rng(n + hub)
    src = np.arange(1, hub + 1)
    rows = np.concatenate([src, [0], np.arange(1, n)])
    cols = np.concatenate([np.zeros(hub, int), [n - 1], (np.arange(1, n) * 7 + 1) % n])
    keep = rows != cols
    pair = np.unique(rows[keep].astype(np.int64) * n + cols[keep])
    rp, col, val = _csr(n, pair // n, pair % n, rng)
    _check(sg, O, n, rp, col, val)


# rows that are empty, and entries given more than once (P_ij twice and P_ji)
def test_symmetrize_duplicates(sg, O):
    n, rng = 777, np.random.default_rng(3)
    rows, cols = rng.integers(0, n, 9000), rng.integers(0, n, 9000)
    keep = (rows != cols) & (rows % 5 != 0) & (cols % 5 != 0)
    rows, cols = np.repeat(rows[keep], 2), np.repeat(cols[keep], 2)
    rp, col, val = _csr(n, rows, cols, rng)
    _check(sg, O, n, rp, col, val)


def _check(sg, O, n, rp, col, val):
    with sg.Context(sg.tsneparams(reorder=0)) as ctx:
        ctx.upload_P(sg.CSR(n, rp, col, val), symmetrize=True)
        P = ctx.get_P()
    S = O.symmetrize(O.CSR(n, rp.astype(np.int64), col, val.astype(np.float64)))
    assert np.array_equal(P.rowptr, S.rowptr) and np.array_equal(P.col, S.col)
    # FP64 sums in another order, rounded once to FP32
    assert np.all(np.abs(P.val - S.val) <= 2.0**-24 * S.val * (1 + 1e-6))
