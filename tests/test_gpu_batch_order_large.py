"""The order a large 3-D job of a batch is spread in, made by many work-groups."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-4  # relative, as for the batch's other terms


def _ring(sg, n):
    i = np.arange(n)
    cols = np.sort(np.stack([(i - 1) % n, (i + 1) % n], 1), 1)
    return sg.CSR(n, (np.arange(n + 1) * 2).astype(np.int32), cols.ravel().astype(np.int32),
                  np.full(2 * n, 0.5 / n, np.float32))


# items of 1024 points: one point over, a last item of one, many; the points over
# the whole grid, most of them in one tile, all in the smallest grid
@pytest.mark.parametrize("n", [1024, 1025, 40001])
@pytest.mark.parametrize("kind", ["wide", "crowd", "start"])
def test_batch_order_of_many_items(sg, O, n, kind):
    rng = np.random.default_rng(n)
    Y = rng.uniform(-15, 15, (n, 3))
    if kind == "crowd":
        Y[n // 20:] = 0.3 * rng.standard_normal((n - n // 20, 3))
    if kind == "start":
        Y = 1e-4 * rng.standard_normal((n, 3))
    with sg.Batch(sg.tsneparams(d=3, reorder=0), 4, 90_000, 400_000) as B:
        # a neighbour on each side, so that the order's rows are not the first
        other = B.add(_ring(sg, 700), symmetrize=False, y_in=rng.uniform(-5, 5, (700, 3)).astype(np.float32), max_iter=50)
        j = B.add(_ring(sg, n), symmetrize=False, y_in=Y.astype(np.float32), max_iter=50)
        B.add(_ring(sg, 300), symmetrize=False, y_in=rng.uniform(-5, 5, (300, 3)).astype(np.float32), max_iter=50)
        for steps in (1, 2, 17):  # admission, the first order, past its renewal
            B.step(steps)
            for job in (other, j):
                Yc = B.get_Y(job).astype(np.float64)
                _, Fr, Z, ng = B.terms(job)
                Fo, Zo, ngo = O.repulsive_interp(Yc, 1.2, O.ZETA_DIRECT)
                assert ng == ngo and np.linalg.norm(Fr - Fo) <= TOL * np.linalg.norm(Fo) and abs(Z - Zo) <= TOL * Zo
