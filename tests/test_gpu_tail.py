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


def entering(ps, p, depth, cache=None):
    """Paths that enter bounce round `depth` of a pass, as the rounds count them."""
    n = []
    for d in (depth, depth + 1):
        q = rrhip.RenderParams.make(max_depth=d, rr_start=p.rr_start, samples_per_pass=p.samples_per_pass)
        n.append(render(ps, q, False, True, cache=cache)[2])
    return n[1] - n[0]


# more paths than the tails of rounds 4, 8 and 12 take (roulette starts
# late): the tail of round 16 takes them all, about 30 to 100 a wave
@pytest.mark.parametrize("width,height,spp,depth,rr_start", [(257, 256, 1, 17, 64), (400, 300, 1, 24, 64),
                                                             (300, 230, 3, 64, 18)])
@pytest.mark.parametrize("film", [False, True])
def test_cloud_tail_takes_any_number_of_paths(width, height, spp, depth, rr_start, film):
    s = scenes.cloud_room(width, height, n=16, sigma_s=(20.0,) * 3, sigma_a=(0.0,) * 3)
    p = rrhip.RenderParams.make(max_depth=depth, rr_start=rr_start, samples_per_pass=spp)
    with rrhip.Context(0) as ctx:
        ps = rrhip.PtScene(ctx, s.desc())
        assert entering(ps, p, 16) > 65536
        ref = render(ps, p, film, True, passes=3)
        for mode in (0, 1, 2):
            same(render(ps, p, film, False, mode, passes=3), ref)
        ps.close()


@pytest.mark.parametrize("width,height,depth", [(300, 230, 17), (320, 240, 40)])
def test_cache_tail_takes_any_number_of_paths(width, height, depth):
    s = scenes.box_room(width, height)
    p = rrhip.RenderParams.make(max_depth=depth, rr_start=64, samples_per_pass=2)
    cfg = rrhip.NrcConfig.make(log2_table=14, train_paths=2048, batch=1024, spread=1e4)
    with rrhip.Context(0) as ctx:
        ps = rrhip.PtScene(ctx, s.desc())
        # some paths have ended in a cache query by then, others do so in the tail
        assert 65536 < entering(ps, p, 16, cfg) < 0.9 * (2 * width * height + 2048)
        same(render(ps, p, False, False, passes=3, cache=cfg), render(ps, p, False, True, passes=3, cache=cfg))
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
