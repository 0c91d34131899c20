"""The CG launched operator by operator (scenes of more than 65,536 particles,
whose solve is not one launch) where the small scenes of the other tests do not
reach: the Project reading that zeroes nodes inside planes, EOS fluid, several
materials in 2D.  One substep against the FP64 oracle to the one-substep bar,
1e-5 relative L2, launched and replayed.
"""
import os

import numpy as np
import pytest

import non_ficks_diffusion_amd as M
import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


def check(d, x, v, m, dt, material=None):
    assert len(m) > 65536
    o = O.Oracle(d, 8, min(os.cpu_count() or 1, 16), O.DOT_FP64 | O.SVD_FP64)
    o.set_particles(x, v, m, material=material)
    o.initialize()
    o.advance_step(dt)
    want = o.particles()
    assert o.cg_stats()["cg_iterations"] > 2
    for graph in (False, True):
        s = M.Scene(d, len(m))
        s.upload(x, v, m, material=material)
        s.initialize()
        s.use_graph(graph)
        s.substep(dt)
        got = s.download()
        s.close()
        assert np.array_equal(got["ids"], want["ids"])
        for k in ("x", "v", "F", "Jp"):
            assert rel(got[k], want[k]) < 1e-5, (graph, k)


def test_project_zero_inside_planes():
    d, x, v, m = M.scene_generate("avalanche", 128, 0, 70000)
    d.project_mode = 0
    d.cg_max_iterations = 20
    v = (v + np.array([-1.0, -0.6, 0.1], np.float32) * (0.5 + x)).astype(np.float32)
    check(d, x, v, m, 0.3 * float(d.max_dt))


def many(name, counts, times, jitter):
    """A preset's particles `times` over, each displaced, of as much mass in all."""
    d, x, v, m = M.scene_generate(name, counts, 0)
    r = np.random.default_rng(3)
    x = (np.tile(x, (times, 1)) + r.uniform(-jitter, jitter, (times * len(x), d.dim))).astype(np.float32)
    x = np.clip(x, 2.0 / counts, 1 - 2.0 / counts)
    v = (np.tile(v, (times, 1)) + 0.5 * (x - 0.5)).astype(np.float32)
    d.cg_max_iterations = 50
    return d, x, v, np.tile(m / times, times).astype(np.float32)


def test_fluid():
    d, x, v, m = many("ref3d_test19", 64, 4, 0.5 / 64)
    check(d, x, v, m, 0.2 * float(d.max_dt))


def test_two_materials_in_2d():
    d, x, v, m = many("ref2d_test16", 256, 23, 1.0 / 256)
    mat = np.tile(M.scene_materials("ref2d_test16", 256, 0), 23)
    check(d, x, v, m, 0.2 * float(d.max_dt), material=mat)
