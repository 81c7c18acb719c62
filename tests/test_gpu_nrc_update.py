"""The cache's one-launch parameter update (no moving average) against the
separate reduction, Adam and packing launches that a moving average takes:
both step the same parameters, so they must agree bit for bit."""
import numpy as np
import pytest

import rrhip

pytestmark = pytest.mark.gpu


def queries(rng, n):
    pos = rng.uniform(-1.2, 1.2, (n, 3))
    pos[0] = 1.0  # the box's last corner
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return rrhip.nrc_queries(pos, d, -d, rng.uniform(0, 1, n), rng.uniform(0, 1, (n, 3)))


# tables of 2^8 (smallest; one dense level of an odd number of entries) and
# 2^14; one, an odd number of, and all levels; batches around the training
# block of 64; epsilon 0, where untouched parameters become 0 / 0
@pytest.mark.parametrize("levels,log2_table,n,eps", [(1, 8, 1, 1e-15), (3, 8, 63, 1e-15), (16, 14, 65, 1e-15),
                                                     (16, 14, 1000, 1e-8), (5, 10, 64, 0.0)])
def test_update_equals_the_separate_launches(levels, log2_table, n, eps):
    rng = np.random.default_rng(levels * 100 + n)
    batches = [(queries(rng, n), rng.uniform(0, 1, (n, 3)).astype(np.float32)) for _ in range(4)]
    probe = queries(rng, 200)
    with rrhip.Context(0) as ctx:
        got = []
        for ema in (0.0, 0.5):
            c = rrhip.Nrc(ctx, rrhip.NrcConfig.make(levels=levels, log2_table=log2_table, base_res=4.0, max_res=160.0,
                                                    lo=(-1.0,) * 3, hi=(1.0,) * 3, batch=4096, seed=3, epsilon=eps,
                                                    ema=ema))
            start = c.get_params()[1]
            for k, (q, t) in enumerate(batches):
                if k == 2:
                    c.gradients(q, t)  # leaves neither a gradient nor a mark behind
                c.train_step(q, t)
            got.append(c.get_params())
            assert c.info()["steps"] == 4
            if ema == 0.0:
                y = c.infer(probe)  # through the bf16 copies the update wrote
                c2 = rrhip.Nrc(ctx, rrhip.NrcConfig.make(levels=levels, log2_table=log2_table, base_res=4.0,
                                                         max_res=160.0, lo=(-1.0,) * 3, hi=(1.0,) * 3, batch=4096))
                c2.set_params(*got[0])
                assert np.array_equal(y, c2.infer(probe), equal_nan=True)
                c2.close()
            c.close()
        for a, b in zip(*got):
            assert np.array_equal(a, b, equal_nan=eps == 0.0)
        assert not np.array_equal(got[0][1], start)
