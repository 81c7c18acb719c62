"""The host build of a path-tracing scene (rrhip_build_info runs it without
a device): instance hierarchies, their bounds and their stack need."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

NO_THREADS = """
#include <errno.h>
#include <pthread.h>
int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) { return EAGAIN; }
"""

BUILD = """
import ctypes, sys
sys.path[:0] = [{root!r} + "/render.rs_amd", {root!r} + "/oracle"]
import numpy as np, rrhip, scenes
rng = np.random.default_rng(1)
s = scenes.Scene(64, 48, 45.0, eye=(0, 0, -30), look_at=(0, 0, 0))
mesh = s.add_mesh(rng.uniform(-1, 1, (300, 3)).astype(np.float32), np.arange(300, dtype=np.uint32).reshape(-1, 3))
m = s.add_material(scenes.matte((0.5, 0.5, 0.5)))
for _ in range(2000):
    s.add_instance(mesh, m, np.hstack([scenes.random_rotation(*rng.uniform(0, 1, 3)), rng.uniform(-9, 9, (3, 1))]))
i = rrhip.SceneInfo()
status = rrhip.load().rrhip_build_info(ctypes.byref(s.desc()), ctypes.byref(i))
print(status, i.num_nodes, i.depth, list(i.bounds_lo), list(i.bounds_hi))
"""


def run_build(**env):
    r = subprocess.run([sys.executable, "-c", BUILD.format(root=ROOT)], capture_output=True, text=True, timeout=300,
                       env={**os.environ, "OPENBLAS_NUM_THREADS": "1", **env})
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout.split("\n")[-2]


def test_build_without_threads(tmp_path):
    """A process that may start no more threads builds the same scene: a
    failed thread start must not leave the library as an exception."""
    src, lib = tmp_path / "no_threads.c", tmp_path / "no_threads.so"
    src.write_text(NO_THREADS)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    want = run_build()
    assert want.startswith("0 ")
    assert run_build(LD_PRELOAD=str(lib)) == want
