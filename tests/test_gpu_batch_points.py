"""Jobs whose points are not numbers, given to a batch next to sound ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _points(n, dim, seed):
    rng = np.random.default_rng(seed)
    c = rng.normal(0, 4, (5, dim))
    return (c[rng.integers(0, 5, n)] + rng.standard_normal((n, dim))).astype(np.float32)


# the filtered search, its exact rows only (few points), and more dimensions
# than the filter takes; a NaN leaves that point, or every point, without rows
@pytest.mark.parametrize("n,dim,where", [(900, 12, 0), (900, 12, 899), (50, 12, 25), (300, 150, 7)])
@pytest.mark.parametrize("d", [2, 3])
def test_nan_point_is_refused(sg, n, dim, where, d):
    X = _points(n, dim, n + dim)
    X[where, dim // 2] = np.nan
    sound = _points(700, 12, 3)
    y0 = (1e-4 * np.random.default_rng(1).standard_normal((700, d))).astype(np.float32)

    def run(with_nan):
        with sg.Batch(sg.tsneparams(d=d), 4, 8000, 800_000) as B:
            j = B.add_points(sound, k=30, u=10.0, y_in=y0, max_iter=20)
            B.step(5)
            if with_nan:
                with pytest.raises(sg.Numeric, match="-4"):
                    B.add_points(X, k=20, u=8.0, max_iter=20)
                t = B.add_points_async(X, k=20, u=8.0, max_iter=20)
                with pytest.raises(sg.Numeric, match="-4"):
                    B.poll_points(t, wait=True)
                assert B.info()["jobs"] == 1
            B.step(16)
            return B.get_Y(j)

    assert np.array_equal(run(True), run(False))
