"""Instance traversal over every kind of placement: tight world bounds, one
instance per TLAS leaf, leaves of every size. First hits (normal, depth, id,
coverage) are functions of the camera sample, which the oracle's brute
two-level traversal draws from the same stream, so they agree to f32
precision on all but silhouette pixels (bars of test_gpu_film.py)."""
import numpy as np
import pytest

import orc
import rrhip
import scenes

from test_gpu_film import first_hit_agree

pytestmark = pytest.mark.gpu

W = H = 48
SPP = 4


def placement(kind, rng):
    r = scenes.random_rotation(*rng.uniform(0, 1, 3))
    if kind == "similar":
        m = r * rng.uniform(0.3, 1.2)
    elif kind == "mirrored":
        m = r @ np.diag([-0.7, 0.5, 0.9])
    else:  # sheared and stretched
        m = r @ (np.diag(rng.uniform(0.2, 1.5, 3)) + np.triu(rng.uniform(-0.8, 0.8, (3, 3)), 1))
    return m


def check(ctx, s, label, max_leaf=4):
    d = s.desc(max_leaf=max_leaf)
    p = rrhip.RenderParams.make(max_depth=1)
    ps = rrhip.PtScene(ctx, d)
    se = ps.session(p)
    se.set_film(True)
    se.render(0, SPP)
    g = se.film()
    se.close()
    ps.close()
    first_hit_agree(g, orc.render_film(d, p, 0, SPP), SPP, label)


def film(ctx, d, p):
    ps = rrhip.PtScene(ctx, d)
    se = ps.session(p)
    se.set_film(True)
    se.render(0, SPP)
    g = se.film()
    se.close()
    ps.close()
    return g


def agree(g, o, normal, depth, label):
    """first_hit_agree with bars of one's own for normals and (relative) depth."""
    bad = (g[:, 16] != o[:, 16]) | (np.abs(g[:, 17] - o[:, 17]) >= 0.5 / SPP) | \
        (np.abs(g[:, 9:15] - o[:, 9:15]).max(1) >= normal) | \
        (np.abs(g[:, 15] - o[:, 15]) > depth * np.maximum(o[:, 15], 1.0))
    assert bad.mean() <= 0.03, f"{label}: {bad.sum()} of {len(bad)} pixels differ"
    assert (o[:, 17] > 0).mean() > 0.02  # something is seen


@pytest.mark.parametrize("kind", ["similar", "mirrored", "sheared"])
@pytest.mark.parametrize("count,offset", [(1, 0.0), (2, 0.0), (61, 0.0), (61, 60.0)])
def test_placements(ctx, kind, count, offset):
    rng = np.random.default_rng(5)
    o = np.array([offset, -offset, 0.5 * offset])
    s = scenes.Scene(W, H, 50.0, eye=tuple(o + (0, 0, -9)), look_at=tuple(o), background=(0.2, 0.3, 0.4))
    pos, idx, nrm = rrhip.gen_icosphere(3, 2)
    mesh = s.add_mesh(pos, idx, nrm)
    for k in range(count):
        t = o + rng.uniform(-3.0, 3.0, 3)
        m = s.add_material(scenes.matte((0.5, 0.4, 0.3), object_id=k + 1))
        s.add_instance(mesh, m, np.hstack([placement(kind, rng), t[:, None]]))
    check(ctx, s, f"{count} {kind} instances at {offset}")


@pytest.mark.parametrize("tris", [1, 2, 3, 4, 5, 8, 9, 33])
@pytest.mark.parametrize("max_leaf", [1, 4, 8])
def test_leaf_sizes(ctx, tris, max_leaf):
    rng = np.random.default_rng(tris)
    s = scenes.Scene(W, H, 50.0, eye=(0, 0, -6), look_at=(0, 0, 0))
    pos = rng.uniform(-1, 1, (3 * tris, 3)).astype(np.float32)
    mesh = s.add_mesh(pos, np.arange(3 * tris, dtype=np.uint32).reshape(-1, 3))
    for k in range(7):
        m = s.add_material(scenes.matte((0.5, 0.5, 0.5), object_id=k + 1))
        s.add_instance(mesh, m, np.hstack([placement("similar", rng), rng.uniform(-1.5, 1.5, (3, 1))]))
    check(ctx, s, f"{tris} triangles, leaves of {max_leaf}", max_leaf)


@pytest.mark.parametrize("kind", ["similar", "mirrored", "sheared"])
def test_placements_far_from_the_origin(ctx, kind):
    """Where the f32 mapping of a ray into an instance moves it most: 1,000
    units out, a rounding of an object-space coordinate is 2e-4 of the
    smallest instance's radius."""
    rng = np.random.default_rng(6)
    o = np.array([1000.0, -1000.0, 500.0])
    s = scenes.Scene(W, H, 50.0, eye=tuple(o + (0, 0, -9)), look_at=tuple(o), background=(0.2, 0.3, 0.4))
    pos, idx, nrm = rrhip.gen_icosphere(3, 2)
    mesh = s.add_mesh(pos, idx, nrm)
    for k in range(61):
        m = s.add_material(scenes.matte((0.5, 0.4, 0.3), object_id=k + 1))
        s.add_instance(mesh, m, np.hstack([placement(kind, rng), (o + rng.uniform(-3.0, 3.0, 3))[:, None]]))
    d, p = s.desc(), rrhip.RenderParams.make(max_depth=1)
    g, f = film(ctx, d, p), orc.render_film(d, p, 0, SPP)
    # positions are rounded to 2^-14 in world and, for scales of 0.2 and more,
    # five times that in object space; a displaced sphere's shading normal
    # turns by a few times that over its radius
    agree(g, f, 5e-3, 4e-4, f"61 {kind} instances far out")


@pytest.mark.parametrize("kind", ["similar", "mirrored", "sheared"])
@pytest.mark.parametrize("count", [1, 61, 200])
def test_placed_curves(ctx, kind, count):
    rng = np.random.default_rng(8)
    s = scenes.Scene(W, H, 50.0, eye=(0, 0, -9), look_at=(0, 0, 0), background=(0.2, 0.3, 0.4))
    a = rng.uniform(-1, 1, (40, 4)) * (1, 1, 1, 0) + (0, 0, 0, 0.08)
    b = a + rng.normal(0, 0.4, (40, 4)) * (1, 1, 1, 0) - (0, 0, 0, 0.03)
    c = s.add_curves(a, b)
    for k in range(count):
        m = s.add_material(scenes.matte((0.5, 0.4, 0.3), object_id=k + 1))
        s.add_instance(c, m, np.hstack([placement(kind, rng), rng.uniform(-3.0, 3.0, (3, 1))]), curves=True)
    d = s.desc()
    g = film(ctx, d, rrhip.RenderParams.make(max_depth=2))
    f = orc.render_film(d, rrhip.RenderParams.make(max_depth=2, ray_offset=1e-9), 0, SPP)
    agree(g, f, 2e-3, 2e-5, f"{count} {kind} curve sets")  # bars of test_gpu_hair.py


@pytest.mark.parametrize("kind", ["similar", "mirrored", "sheared"])
@pytest.mark.parametrize("count", [1, 61, 200])
def test_placed_deforming_meshes(ctx, kind, count):
    rng = np.random.default_rng(9)
    s = scenes.Scene(W, H, 50.0, eye=(0, 0, -9), look_at=(0, 0, 0), background=(0.2, 0.3, 0.4))
    pos, idx, _ = rrhip.gen_icosphere(3, 2)
    mesh = s.add_mesh(pos, idx, positions1=pos * (1.4, 0.6, 1.0) + (0.3, 0.0, -0.2))
    for k in range(count):
        m = s.add_material(scenes.matte((0.5, 0.4, 0.3), object_id=k + 1))
        s.add_instance(mesh, m, np.hstack([placement(kind, rng), rng.uniform(-3.0, 3.0, (3, 1))]))
    d, p = s.desc(), rrhip.RenderParams.make(max_depth=1)
    first_hit_agree(film(ctx, d, p), orc.render_film(d, p, 0, SPP), SPP, f"{count} {kind} deforming meshes")
