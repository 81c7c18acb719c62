"""Queue appends of the shading pass: one place per block for the next
paths and the shadow records. A session's image must not depend on how its
paths fall into blocks, so at path counts around the block and wave sizes
it equals the persistent batch launch's, which has no queues."""
import numpy as np
import pytest

import rrhip
import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,spp", [(1, 1, 1), (63, 1, 1), (64, 1, 1), (5, 13, 1), (85, 3, 1), (16, 16, 1),
                                              (257, 1, 1), (67, 43, 3)])
@pytest.mark.parametrize("cloud", [False, True])
def test_session_equals_persistent_batch(width, height, spp, cloud):
    s = scenes.cloud_room(width, height, n=16) if cloud else scenes.box_room(width, height)
    p = rrhip.RenderParams.make(max_depth=8, samples_per_pass=spp)
    with rrhip.Context(0) as ctx:
        ps = rrhip.PtScene(ctx, s.desc())
        se = ps.session(p)
        se.render(0, spp)
        a = se.accum()
        st = se.stats()
        b = rrhip.Batch(ctx, [(ps, spp, p)])
        b.render_persistent()
        assert np.array_equal(a, b.accum(0))
        bs = b.stats()
        assert (st["extension_rays"], st["shadow_rays"]) == (bs["extension_rays"], bs["shadow_rays"])
        b.close()
        se.close()
        ps.close()
