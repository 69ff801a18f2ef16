"""The Morton re-order of a running job where it pays: taken, and exact in the caller's order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-4  # relative, as for the single job's other terms


def _lattice(side, rng):
    """Points of a lattice in random order, tied to their eight neighbours and to one of n / 200 points
    picked at random: a breadth-first order of it is no order in the plane."""
    n = side * side
    name = rng.permutation(n)  # lattice position -> index
    x, y = np.divmod(np.arange(n), side)
    rows, cols = [], []
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            u, v = x + dx, y + dy
            ok = (u >= 0) & (u < side) & (v >= 0) & (v < side) & ((dx != 0) | (dy != 0))
            rows.append(name[np.arange(n)[ok]])
            cols.append(name[(u * side + v)[ok]])
    hub = rng.integers(0, n // 200, n)
    rows += [np.arange(n), hub]
    cols += [hub, np.arange(n)]
    pair = np.unique(np.concatenate(rows).astype(np.int64) * n + np.concatenate(cols))
    r, c = pair // n, pair % n
    r, c = r[r != c], c[r != c]
    rp = np.zeros(n + 1, np.int64)
    np.add.at(rp, r + 1, 1)
    Y = np.empty((n, 2), np.float32)
    Y[name] = 0.03 * (np.stack([x, y], 1) + 0.2 * rng.standard_normal((n, 2)))
    return np.cumsum(rp), c.astype(np.int32), np.full(c.size, 1.0 / c.size, np.float32), Y


def test_reorder_applied(sg, O):
    # 1.69 M points, whose gathers leave the cache in the order of P: 0.19 ms per
    # evaluation, 0.13 along the curve, so the comparison accepts it every time
    rng = np.random.default_rng(12)
    rp, col, val, Y0 = _lattice(1300, rng)
    n = Y0.shape[0]
    So = O.CSR(n, rp, col, val.astype(np.float64))

    def check(ctx):
        Y = ctx.get_Y().astype(np.float64)
        Fa, Fr, Z, ng = ctx.terms()
        Fao = O.attractive(So, Y)
        Fro, Zo, ngo = O.repulsive_interp(Y.copy(), 0.7, O.ZETA_DIRECT)
        assert ng == ngo and abs(Z - Zo) <= TOL * Zo
        assert np.linalg.norm(Fa - Fao) <= TOL * np.linalg.norm(Fao)
        assert np.linalg.norm(Fr - Fro) <= TOL * np.linalg.norm(Fro)

    with sg.Context(sg.tsneparams(reorder=2)) as ctx:
        ctx.upload_P(sg.CSR(n, rp, col, val), symmetrize=False)
        ctx.set_Y(Y0)
        ctx.step(50)
        assert ctx.reorders()["applied"] == 0
        before = ctx.get_Y()
        kl = ctx.kl(1.0)
        ctx.step(1)
        assert ctx.reorders()["applied"] == 1
        # one iteration moves no point far: the rows are still the caller's
        after = ctx.get_Y()
        assert np.linalg.norm(after - before) < 0.05 * np.linalg.norm(before)
        check(ctx)
        # Y given again without resetting the optimiser, and read back
        ctx.set_Y(before, reset_state=False)
        back = ctx.get_Y()
        assert np.abs(back - (before - before.astype(np.float64).mean(0))).max() <= 1e-5 * np.abs(before).max()
        assert abs(ctx.kl(1.0) - kl) <= 1e-6 * abs(kl)
        check(ctx)
        ctx.step(5)
        check(ctx)
        P = ctx.get_P()
        assert np.array_equal(P.rowptr, rp) and np.array_equal(P.col, col) and np.array_equal(P.val, val)
