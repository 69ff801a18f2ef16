"""The phase times of a context against the attractive kernel timed by itself."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# points enough that the centring takes a fifth of a short attractive term: it
# belongs to the update, not to the next iteration's attractive phase
def test_centring_is_not_in_the_attractive_phase(sg):
    n, iters = 3_000_000, 12
    i = np.arange(n)
    P = sg.CSR(n, np.arange(n + 1) * 2, np.sort(np.stack([(i - 1) % n, (i + 1) % n], 1), 1).ravel().astype(np.int32),
               np.full(2 * n, 0.5 / n, np.float32))
    Y = (1e-4 * np.random.default_rng(0).standard_normal((n, 3))).astype(np.float32)
    with sg.Context(sg.tsneparams(d=3, reorder=0)) as ctx:
        ctx.upload_P(P, symmetrize=False)
        alone = min(ctx.tuning()["candidates_ms"])
        # the tuner's usual choice; the plain form is level with it only while Y is warm
        # in cache, as it is between the tuner's launches (0.161 ms; 0.201 in an iteration)
        ctx.set_attractive(16, 2, 128)
        ctx.set_Y(Y)
        ctx.step(2)
        best = 1e9
        for _ in range(3):
            ctx.step(iters)
            t = ctx.timing()
            best = min(best, t[0] / iters)
            assert t[6] == iters and abs(t[:5].sum() - t[5]) <= 1e-9 * t[5] and (t[:5] > 0).all()
    # the kernel, a launch before it, and a tenth (with the centring in it 0.184 against 0.161)
    assert best <= 1.1 * alone + 0.004
