"""COO and hybrid attractive kernels at the edges of their runs, against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-5  # FP32 sums of up to 3000 terms: below 3000 * 2^-24 / sqrt(3000) of their size


@pytest.fixture(scope="module")
def sg():
    import sgtsne_amd

    return sgtsne_amd


@pytest.fixture(scope="module")
def O():
    from oracle import oracle

    return oracle


def _matrix(kind, n, rng):
    """Symmetric patterns whose rows end inside lanes, fill them, and span waves."""
    if kind == "single":  # rows of one entry: every entry ends a run
        i = np.arange(n)
        rows, cols = i, i ^ 1
    elif kind == "hub":  # one row of n - 1 entries (many waves), the others of one
        rows = np.concatenate([np.zeros(n - 1, int), np.arange(1, n)])
        cols = np.concatenate([np.arange(1, n), np.zeros(n - 1, int)])
    else:  # ragged rows, some of them empty
        dense = rng.random((n, n)) < np.minimum(0.9, rng.pareto(1.0, n) * 0.02)[:, None]
        dense[::7] = False
        dense[:, ::7] = False
        dense |= dense.T
        np.fill_diagonal(dense, False)
        rows, cols = np.nonzero(dense)
    order = np.lexsort((cols, rows))
    rows, cols = rows[order], cols[order]
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, rows + 1, 1)
    val = np.full(rows.size, 1.0 / rows.size)
    return np.cumsum(rp), cols.astype(np.int32), val


@pytest.mark.parametrize("fmt,width", [("COO", 0), ("HYBRID", 0), ("HYBRID", 1), ("HYBRID", 33)])
@pytest.mark.parametrize("kind,n,d", [("single", 514, 2), ("hub", 3000, 1), ("ragged", 257, 3), ("ragged", 640, 2)])
def test_attractive_runs(sg, O, fmt, width, kind, n, d):
    rng = np.random.default_rng(n + d)
    rp, col, val = _matrix(kind, n, rng)
    Y = (rng.standard_normal((n, d)) * 3).astype(np.float32)
    prm = sg.tsneparams(d=d, format=getattr(sg, "FORMAT_" + fmt), ell_width=width, reorder=0)
    with sg.Context(prm) as ctx:
        ctx.upload_P(sg.CSR(n, rp, col, val), symmetrize=False)
        ctx.set_Y(Y)
        Fa = ctx.terms()[0]
        Yc = ctx.get_Y().astype(np.float64)
    ref = O.attractive(O.CSR(n, rp.astype(np.int64), col, val.astype(np.float32).astype(np.float64)), Yc)
    assert np.linalg.norm(Fa - ref) <= TOL * np.linalg.norm(ref)


# grids that go through the tile order and the fixed-point windows: points that
# end a batch of 4096, one crowded tile, every point on the box's faces
@pytest.mark.parametrize("d,n,kind", [(2, 4096, "wide"), (2, 4097, "crowd"), (2, 9000, "faces"), (3, 4095, "wide"),
                                      (3, 8193, "crowd"), (3, 5000, "faces")])
def test_large_grid_order(sg, O, d, n, kind):
    rng = np.random.default_rng(7 * n + d)
    R = 40.0 if d == 2 else 20.0
    Y = rng.uniform(-R, R, (n, d))
    if kind == "crowd":
        Y[n // 10:] = 0.3 * rng.standard_normal((n - n // 10, d)) + 5.0
    elif kind == "faces":
        Y[np.arange(n), rng.integers(0, d, n)] = R * rng.choice([-1, 1], n)
    Y = Y.astype(np.float32)
    i = np.arange(n)
    P = sg.CSR(n, np.arange(n + 1), i[::-1], np.full(n, 1.0 / n))
    with sg.Context(sg.tsneparams(d=d, reorder=0)) as ctx:
        ctx.upload_P(P, symmetrize=True)
        ctx.set_Y(Y)
        _, Fr, Z, ng = ctx.terms()
        Yc = ctx.get_Y().astype(np.float64)
        again = ctx.terms()
    assert ng > (73 if d == 2 else 16)
    Fo, Zo, ngo = O.repulsive_interp(Yc.copy(), 0.7 if d == 2 else 1.2, O.ZETA_DIRECT)
    # FP32 grids and transforms against FP64: the single-precision bar of the other term tests
    assert ng == ngo and abs(Z - Zo) <= 1e-4 * Zo and np.linalg.norm(Fr - Fo) <= 1e-4 * np.linalg.norm(Fo)
    assert np.array_equal(Fr, again[1]) and Z == again[2]


# the small grids: work-groups of one short, full and one long round of points,
# fixed sides below 16, both Z modes
@pytest.mark.parametrize("zeta", ["DIRECT", "ALGEBRAIC"])
@pytest.mark.parametrize("d,n,ng_fixed", [(2, 255, 0), (2, 3000, 25), (2, 700, 6), (3, 255, 0), (3, 257, 0), (3, 32769, 0), (3, 900, 9)])
def test_small_grids(sg, O, d, n, ng_fixed, zeta):
    rng = np.random.default_rng(n + d)
    Y = (1.5 * rng.standard_normal((n, d))).astype(np.float32)
    i = np.arange(n)
    P = sg.CSR(n, np.arange(n + 1), i[::-1], np.full(n, 1.0 / n))
    prm = sg.tsneparams(d=d, reorder=0, zeta_mode=getattr(sg, "ZETA_" + zeta))
    if ng_fixed:
        prm.grid_mode, prm.ng = sg.GRID_FIXED, ng_fixed
    with sg.Context(prm) as ctx:
        ctx.upload_P(P, symmetrize=True)
        ctx.set_Y(Y)
        _, Fr, Z, ng = ctx.terms()
        Yc = ctx.get_Y().astype(np.float64)
    Fo, Zo, ngo = O.repulsive_interp(Yc.copy(), 0.7 if d == 2 else 1.2, getattr(O, "ZETA_" + zeta), ng_fixed)
    # FP32 against FP64, the single-precision bar of the other term tests; the
    # algebraic Z cancels N |y|^2-sized terms of FP32 potentials: ten times it
    tz = 1e-4 if zeta == "DIRECT" else 1e-3
    assert ng == ngo and abs(Z - Zo) <= tz * abs(Zo)
    assert np.linalg.norm(Fr * Z - Fo * Zo) <= 1e-4 * np.linalg.norm(Fo * Zo)
