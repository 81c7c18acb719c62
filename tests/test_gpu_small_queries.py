"""Ray batches too small to fill the device run with 4, 8, 16 or 32 lanes a
wave; hits must be those of whole wavefronts (64 rays a wave, set by hand)
and of the oracle."""
import numpy as np
import pytest

import orc
import rrhip

pytestmark = pytest.mark.gpu


def test_small_batches_equal_whole_wavefronts():
    pos, idx = rrhip.gen_heightfield(60, 31, 7)
    m = orc.Mesh(pos, idx, bins=32, max_leaf=4, sah_leaf_mult=1)
    # around the wave, and on both sides of where each lane count ends for
    # 6,144 wave slots
    sizes = [1, 3, 4, 5, 63, 64, 65, 257, 9001, 12288, 12289, 24577, 49153, 65537, 98305, 131073, 200003]
    rays = rrhip.gen_query_rays(pos.min(0), pos.max(0), 0.1, 3, max(sizes))
    op, ot, _, _ = m.trace_closest(rays)
    with rrhip.Context(0) as ctx:
        sc = ctx.upload_mesh(pos, idx)
        t = sc.get_tuning()
        got = [(sc.trace_closest(rays[:n]), sc.trace_any(rays[:n])) for n in sizes]
        sc.set_tuning(t["block"], t["stack"], 64, t["width"])
        for n, (hits, occ) in zip(sizes, got):
            ref = sc.trace_closest(rays[:n])
            assert hits.tobytes() == ref.tobytes(), n
            assert np.array_equal(occ, sc.trace_any(rays[:n])), n
            hit = op[:n] != rrhip.NO_HIT
            assert np.array_equal(occ.astype(bool), hit), n
            assert np.array_equal(hits["t"][hit], ot[:n][hit].astype(np.float32)), n
        sc.close()
