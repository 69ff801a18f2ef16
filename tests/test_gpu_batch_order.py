"""3-D jobs of a batch, spread along the tiles of their grids, against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-4  # relative, per job and iteration, as for the batch's other terms


@pytest.fixture(scope="module")
def sg():
    import sgtsne_amd

    return sgtsne_amd


@pytest.fixture(scope="module")
def O():
    from oracle import oracle

    return oracle


def _ring(sg, O, n):
    """Each point tied to the next two: a symmetric P of any size."""
    i = np.arange(n)
    cols = np.sort(np.stack([(i + s) % n for s in (-2, -1, 1, 2)], 1), 1)
    rp = np.arange(n + 1) * 4
    val = np.full(4 * n, 1.0 / (4 * n))
    return (sg.CSR(n, rp.astype(np.int32), cols.ravel().astype(np.int32), val.astype(np.float32)),
            O.CSR(n, rp.astype(np.int64), cols.ravel().astype(np.int32), val.astype(np.float32).astype(np.float64)))


def _check(B, O, jobs, h=1.2):
    for j, So in jobs:
        Y = B.get_Y(j).astype(np.float64)
        Fa, Fr, Z, _ = B.terms(j)
        Fro, Zo, _ = O.repulsive_interp(Y.copy(), h, O.ZETA_DIRECT)
        assert np.linalg.norm(Fa - O.attractive(So, Y)) <= TOL * np.linalg.norm(O.attractive(So, Y))
        assert np.linalg.norm(Fr - Fro) <= TOL * np.linalg.norm(Fro)
        assert abs(Z - Zo) <= TOL * Zo


# sizes at the edges of an item (256) and of the ordering work-group (1024), none
# so small that it leaves its grid within 20 steps; extents from one tile per axis to more than 16 of 4 cells
@pytest.mark.parametrize("sizes,extent", [((255, 256, 257), 2.0), ((256, 1023, 1025), 30.0), ((1024, 2049, 300), 60.0)])
def test_batch_order_follows_the_jobs(sg, O, sizes, extent):
    rng = np.random.default_rng(sum(sizes))
    with sg.Batch(sg.tsneparams(d=3), 8, 8000, 200_000) as B:
        jobs = []
        for n in sizes:
            S, So = _ring(sg, O, n)
            jobs.append((B.add(S, symmetrize=False, y_in=rng.uniform(-extent / 2, extent / 2, (n, 3)).astype(np.float32),
                               max_iter=100, ng_cap=128), So))
        B.step(1)
        _check(B, O, jobs)
        B.step(18)  # past the renewal of the order, the points having moved
        _check(B, O, jobs)
        # the first job leaves (the others move down), a new one takes its slot
        B.remove(jobs.pop(0)[0])
        S, So = _ring(sg, O, 777)
        jobs.append((B.add(S, symmetrize=False, y_in=rng.uniform(-extent / 2, extent / 2, (777, 3)).astype(np.float32),
                           max_iter=100, ng_cap=128), So))
        B.step(2)
        _check(B, O, jobs)


# 1-D and 2-D jobs are spread in eighths of an item of 1024 points: items that
# eight does not divide, one of a single point, and one shorter than eight parts
@pytest.mark.parametrize("d,h", [(1, 0.5), (2, 0.7)])
@pytest.mark.parametrize("sizes", [(300, 1025, 1031), (1023, 1024, 2049)])
def test_batch_spread_in_eighths(sg, O, d, h, sizes):
    rng = np.random.default_rng(sum(sizes) + d)
    with sg.Batch(sg.tsneparams(d=d), 4, 8000, 200_000) as B:
        jobs = []
        for n in sizes:
            S, So = _ring(sg, O, n)
            jobs.append((B.add(S, symmetrize=False, y_in=rng.uniform(-15, 15, (n, d)).astype(np.float32), max_iter=100), So))
        B.step(1)
        _check(B, O, jobs, h)
