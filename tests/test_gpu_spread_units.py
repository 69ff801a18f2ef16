"""The runs of points a large grid is spread in, at the edges of their lengths, against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-4  # relative, as for the single job's other terms


@pytest.fixture(scope="module")
def sg():
    import sgtsne_amd

    return sgtsne_amd


@pytest.fixture(scope="module")
def O():
    from oracle import oracle

    return oracle


# runs of 64 points up to 32,768 of them, then 128; a last run of one point; the
# shortest job; a 3-D grid beyond the matrix-core form
@pytest.mark.parametrize("n,d,extent", [(63, 2, 60.0), (4097, 2, 60.0), (32768, 2, 60.0), (32769, 2, 60.0), (4097, 3, 40.0)])
def test_repulsion_run_lengths(sg, O, n, d, extent):
    rng = np.random.default_rng(n + d)
    Y = rng.uniform(-extent / 2, extent / 2, (n, d)).astype(np.float32)
    i = np.arange(n)
    cols = np.sort(np.stack([(i - 1) % n, (i + 1) % n], 1), 1)
    P = sg.CSR(n, (np.arange(n + 1) * 2).astype(np.int32), cols.ravel().astype(np.int32),
               np.full(2 * n, 0.5 / n, np.float32))
    with sg.Context(sg.tsneparams(d=d, reorder=0)) as ctx:
        ctx.upload_P(P, symmetrize=False)
        ctx.set_Y(Y)
        _, Fr, Z, ng = ctx.terms()
        Yc = ctx.get_Y().astype(np.float64)
    Fo, Zo, ngo = O.repulsive_interp(Yc, {2: 0.7, 3: 1.2}[d], O.ZETA_DIRECT)
    assert ng == ngo
    assert np.linalg.norm(Fr - Fo) <= TOL * np.linalg.norm(Fo) and abs(Z - Zo) <= TOL * Zo
