"""Paths finished by one tail launch against bounce rounds to the end (which
profiling keeps): the same paths, so the same bits."""
import numpy as np
import pytest

import rrhip
import scenes

pytestmark = pytest.mark.gpu


def render(ps, p, film, profile, mode=0, passes=1, cache=None):
    se = ps.session(p)
    se.set_launch_mode(mode)
    if film:
        se.set_film(True)
    if profile:
        se.set_profiling(True)
    c = rrhip.Nrc(ps.ctx, cache) if cache else None
    if c:
        se.set_nrc(c)
    out = []
    for k in range(passes):
        se.render(k * p.samples_per_pass, p.samples_per_pass)
        st = se.stats()
        out += [se.accum(), se.film() if film else None, st["extension_rays"], st["shadow_rays"]]
    if c:
        out += list(c.get_params())
        c.close()
    se.close()
    return out


def same(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


# path counts around a wave and the 65,536 paths that end in a tail at most;
# depths that end before, in and after the rounds with a tail (4, 8, 12, 16)
@pytest.mark.parametrize("width,height,spp,depth", [(1, 1, 1, 64), (63, 1, 1, 5), (65, 3, 1, 17), (257, 257, 1, 64),
                                                    (300, 230, 3, 16), (40, 30, 2, 4)])
@pytest.mark.parametrize("film", [False, True])
def test_cloud_tail_equals_rounds(width, height, spp, depth, film):
    s = scenes.cloud_room(width, height, n=16)
    p = rrhip.RenderParams.make(max_depth=depth, samples_per_pass=spp)
    with rrhip.Context(0) as ctx:
        ps = rrhip.PtScene(ctx, s.desc())
        ref = render(ps, p, film, True, passes=3)
        for mode in (0, 1, 2):  # direct, one graph replayed, sorted queue
            same(render(ps, p, film, False, mode, passes=3), ref)
        ps.close()


@pytest.mark.parametrize("width,height,depth", [(9, 7, 20), (320, 210, 12)])
def test_cache_tail_equals_rounds(width, height, depth):
    s = scenes.box_room(width, height)
    p = rrhip.RenderParams.make(max_depth=depth, samples_per_pass=2)
    cfg = rrhip.NrcConfig.make(log2_table=14, train_paths=2048, batch=1024)
    with rrhip.Context(0) as ctx:
        ps = rrhip.PtScene(ctx, s.desc())
        same(render(ps, p, False, False, passes=3, cache=cfg), render(ps, p, False, True, passes=3, cache=cfg))
        ps.close()
