"""The gather through a copy of the grid in LDS, at the number of points it starts from."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-4  # relative, as for the single job's other terms


# one point under the number, that number and one over; the largest 2-D grid it
# takes (side 64) and the 3-D one, both Z modes
@pytest.mark.parametrize("zeta", ["DIRECT", "ALGEBRAIC"])
@pytest.mark.parametrize("d,extent", [(2, 42.0), (2, 12.0), (3, 14.0)])
@pytest.mark.parametrize("n", [199_999, 200_000, 200_001])
def test_gather_of_many_points(sg, O, n, d, extent, zeta):
    rng = np.random.default_rng(n + d)
    Y = rng.uniform(-extent / 2, extent / 2, (n, d)).astype(np.float32)
    i = np.arange(n)
    P = sg.CSR(n, np.arange(n + 1), ((i + 1) % n).astype(np.int32), np.full(n, 1.0 / n, np.float32))
    with sg.Context(sg.tsneparams(d=d, reorder=0, zeta_mode=getattr(sg, "ZETA_" + zeta))) as ctx:
        ctx.upload_P(P, symmetrize=False)
        ctx.set_Y(Y)
        _, Fr, Z, ng = ctx.terms()
        Yc = ctx.get_Y().astype(np.float64)
    assert ng <= (64 if d == 2 else 16)
    Fo, Zo, ngo = O.repulsive_interp(Yc, {2: 0.7, 3: 1.2}[d], getattr(O, "ZETA_" + zeta))
    # the algebraic Z cancels N |y|^2-sized terms of FP32 potentials: ten times the bar
    tz = TOL if zeta == "DIRECT" else 10 * TOL
    assert ng == ngo and abs(Z - Zo) <= tz * abs(Zo)
    assert np.linalg.norm(Fr * Z - Fo * Zo) <= TOL * np.linalg.norm(Fo * Zo)
