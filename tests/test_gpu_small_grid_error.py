"""Forces on the grids whose convolution is a direct sum: no further from 64 bits than with the transforms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# the root mean square error of Frep over three embeddings, as measured with the
# FP32 transforms on the same ones (FP32 sums in place of the FP64 ones exceed it at
# each of these: 1.36e-7, 8.76e-7, 9.51e-7, 8.19e-7)
@pytest.mark.parametrize("d,n,scale,ng,bar", [(2, 700, 1e-4, 16, 1.33e-7), (2, 700, 1.5, 16, 8.42e-7),
                                              (2, 10000, 1.5, 20, 9.18e-7), (3, 10000, 1.5, 16, 8.11e-7)])
def test_direct_sum_error(sg, O, d, n, scale, ng, bar):
    i = np.arange(n)
    P = sg.CSR(n, np.arange(n + 1), i[::-1].astype(np.int32), np.full(n, 1.0 / n, np.float32))
    err = []
    for seed in (1, 2, 3):
        Y = (scale * np.random.default_rng(1000 * seed + n + d).standard_normal((n, d))).astype(np.float32)
        with sg.Context(sg.tsneparams(d=d, reorder=0)) as ctx:
            ctx.upload_P(P)
            ctx.set_Y(Y)
            _, Fr, _, got = ctx.terms()
            Yc = ctx.get_Y().astype(np.float64)
        Fo, _, ngo = O.repulsive_interp(Yc, {2: 0.7, 3: 1.2}[d], O.ZETA_DIRECT)
        assert got == ngo
        if got == ng:
            err.append(np.linalg.norm(Fr - Fo) / np.linalg.norm(Fo))
    assert err and np.sqrt(np.mean(np.square(err))) <= bar
