"""Downloads at the edges of the id tiles, with particles missing.

A download is ordered on the device (tiles of 1024 ids): the particles of a
scene come back by id with their own values bit for bit, whatever order the
binning left them in, and without those that left the domain.
"""
import numpy as np
import pytest

import non_ficks_diffusion_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 5000])
def test_download_is_the_upload_by_id(dim, n):
    r = np.random.default_rng(10 * n + dim)
    d, _, _, _ = M.scene_generate("disk2d" if dim == 2 else "two_balls", 32, 0)
    descs, parts = [d, d], []
    for _ in descs:
        p = dict(x=r.uniform(0.1, 0.9, (n, dim)), v=r.normal(size=(n, dim)), F=r.normal(size=(n, dim, dim)),
                 Jp=r.uniform(0.5, 2, n), mass=r.uniform(0.1, 1, n), volume=r.uniform(0.1, 1, n))
        p = {k: a.astype(np.float32) for k, a in p.items()}
        p["x"][r.random(n) < 0.1] += 2  # outside the domain: dropped by the binning
        parts.append(p)
    b = M.Batch(descs, [n, n + 7])
    for k, p in enumerate(parts):
        b.upload(k, p["x"], p["v"], p["mass"], F=p["F"], Jp=p["Jp"], volume=p["volume"])
    for k, p in enumerate(parts):  # as uploaded
        got = b.download(k)
        assert np.array_equal(got["ids"], np.arange(n))
        for f in p:
            assert np.array_equal(got[f], p[f]), f
    b.initialize()
    for k, p in enumerate(parts):  # binned
        keep = np.nonzero((p["x"] < 1).all(1))[0]
        got = b.download(k)
        assert np.array_equal(got["ids"], keep)
        for f in p:
            assert np.array_equal(got[f], p[f][keep]), f
        assert not got["material"].any()
    if len(keep):
        with pytest.raises(M.MPMError):
            b.download(1, cap=len(keep) - 1)
    b.close()


@pytest.mark.parametrize("dim", [2, 3])
def test_download_with_ids_past_the_capacity(dim):
    """Ids are not reused, so a scene that keeps losing and gaining particles
    passes its capacity: the download then orders on the host, with the same
    result."""
    r = np.random.default_rng(dim)
    d, _, _, _ = M.scene_generate("disk2d" if dim == 2 else "two_balls", 32, 0)
    d.gravity[:] = (0.0,) * len(d.gravity)
    d.nplanes = 0
    dt = float(d.max_dt)
    cap, stay, leave = 200, 10, 50
    s = M.Scene(d, cap)
    mass, x_of, alive = {}, {}, []
    ids = 0
    for step in range(6):
        n = stay + leave
        x = r.uniform(0.3, 0.7, (n, dim)).astype(np.float32)
        v = np.zeros((n, dim), np.float32)
        v[stay:] = 2.0 / dt  # leaves the domain in the substep
        m = r.uniform(0.5, 1.0, n).astype(np.float32)
        x[stay:] = 0.9 + 0.001 * (x[stay:] - 0.5)  # away from those that stay
        if step == 0:
            s.upload(x, v, m)
            s.initialize()
        else:
            s.add_particles(x, v, m)
        mass.update(zip(range(ids, ids + n), m))
        x_of.update(zip(range(ids, ids + n), x))
        alive += range(ids, ids + stay)
        ids += n
        s.substep(dt)
        got = s.download()
        assert got["ids"].tolist() == alive
        assert np.array_equal(got["mass"], np.array([mass[k] for k in alive]))
        assert np.abs(got["x"] - np.array([x_of[k] for k in alive])).max() < 1e-3
        assert np.all(got["volume"] > 0) and not got["material"].any()
        assert np.abs(got["F"] - np.eye(dim)).max() < 0.1 and np.abs(got["Jp"] - 1).max() < 0.1
    assert ids > cap
    with pytest.raises(M.MPMError):
        s.download(cap=len(alive) - 1)
    s.close()
