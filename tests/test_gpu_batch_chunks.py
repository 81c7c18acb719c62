"""The persistent batch launch deals the samples of chunks of whole pixels to
its waves' lanes: at samples per pixel around a chunk's 64 and pixel counts
that leave a remainder, every job equals its own session bit for bit."""
import numpy as np
import pytest
import torch

import rrhip
import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jobs", [[(1, 1, 1)], [(1, 1, 64), (1, 1, 65)], [(5, 13, 1), (3, 7, 33), (9, 5, 5)],
                                  [(17, 3, 64), (5, 5, 65), (7, 1, 130), (64, 1, 2)],
                                  [(200, 101, 3), (2, 2, 63), (61, 67, 16)]])
def test_every_job_equals_its_session(jobs):
    with rrhip.Context(0) as ctx:
        work, rays = [], 0
        for j, (w, h, spp) in enumerate(jobs):
            s = scenes.cloud_room(w, h, n=16, seed=j) if j % 2 else scenes.box_room(w, h)
            p = rrhip.RenderParams.make(max_depth=20 if j % 2 else 6, samples_per_pass=spp, firefly_clamp=2.0)
            work.append((rrhip.PtScene(ctx, s.desc()), spp, p))
        b = rrhip.Batch(ctx, work)
        for _ in range(2):  # the second launch starts from used buffers
            job_ms, total = b.render_persistent()
            assert (job_ms > 0).all() and (job_ms <= total + 1.0).all()
            rays = 0
            for j, (ps, spp, p) in enumerate(work):
                se = ps.session(p)
                se.render(0, spp)
                assert np.array_equal(se.accum(), b.accum(j)), jobs[j]
                rays += se.stats()["extension_rays"]
                se.close()
            assert b.stats()["extension_rays"] == rays
        b.close()
        for ps, _, _ in work:
            ps.close()


@pytest.mark.parametrize("spp,least,most", [(64, 100, 400), (65, 0, 100)])
def test_sample_scratch_only_where_samples_wait(spp, least, most):
    """Jobs of more than 64 samples a pixel add them one by one: the first
    persistent launch of such a batch takes none of the 134 MB in which the
    others' samples wait."""
    s = scenes.box_room(8, 8)
    p = rrhip.RenderParams.make(max_depth=2)
    with rrhip.Context(0) as ctx:
        ps = rrhip.PtScene(ctx, s.desc())
        for first in (True, False):  # the first batch loads the kernel's code
            b = rrhip.Batch(ctx, [(ps, spp, p)])
            free = torch.cuda.mem_get_info(0)[0]
            b.render_persistent()
            taken = (free - torch.cuda.mem_get_info(0)[0]) >> 20
            b.close()
        assert least <= taken <= most, taken
        ps.close()
