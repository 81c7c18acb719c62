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
