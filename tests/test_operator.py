"""The CG operator at the edges of its chunks and cell counts.

A block's particles are taken 256 at a time and its cells are sorted by
count up to 63: one substep of a scene that packs a given number of
particles into one cell (next to a sparse neighbourhood that spans blocks)
must match the FP64 oracle to the one-substep bar, 1e-5 relative L2, per
field.  The particles carry a velocity gradient, so the operator's result
reaches every compared field.
"""
import contextlib
import threading

import numpy as np
import pytest

import non_ficks_diffusion_amd as M
import oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 63, 64, 255, 256, 257, 513, 700])
def test_cell_and_chunk_edges(dim, n):
    r = np.random.default_rng(100 * dim + n)
    name, counts = ("disk2d", 32) if dim == 2 else ("two_balls", 32)
    d, _, _, _ = M.scene_generate(name, counts, 0)
    d.cg_max_iterations = 200
    dx = 1.0 / counts
    # n particles in cell 15 of every axis, the last of its block in 2D and 3D
    cell = (15 + r.uniform(0.02, 0.98, (n, dim))) * dx
    # two per cell over the six cells around it (several blocks, sparse cells)
    g = np.stack(np.meshgrid(*[np.arange(12, 18)] * dim, indexing="ij"), -1).reshape(-1, dim)
    around = (np.repeat(g, 2, axis=0) + r.uniform(0.1, 0.9, (2 * len(g), dim))) * dx
    x = np.concatenate([cell, around]).astype(np.float32)
    # a rate of about one per second, with shear
    v = ((x - 0.5) @ r.uniform(-1.0, 1.0, (dim, dim)) + 0.5).astype(np.float32)
    m = np.full(len(x), 400.0 * dx ** dim / 8, np.float32)
    dt = 0.5 * float(d.max_dt)
    s = M.Scene(d, len(m))
    s.upload(x, v, m)
    s.initialize()
    st = s.substep(dt, stats=True)
    got = s.download()
    s.close()
    o = O.Oracle(d, 8, 4, O.DOT_FP64 | O.SVD_FP64)
    o.set_particles(x, v, m)
    o.initialize()
    o.advance_step(dt)
    want = o.particles()
    assert st["cg_converged"] == 1
    assert np.array_equal(got["ids"], want["ids"])
    for k in ("x", "v", "F", "Jp"):
        assert rel(got[k], want[k]) < 1e-5, k


# active blocks (all scenes) of the scattered particles below: 322, 606 (a pair of
# blocks per work-group), 1271; 638 and 1741 for two and three scenes of a batch
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("scenes,n,blocks", [(1, 100, 322), (1, 200, 606), (1, 700, 1271), (2, 100, 638), (3, 200, 1741)])
def test_solve_by_number_of_blocks(scenes, n, blocks, graph):
    """Scattered particles make hundreds of active blocks of a few hundred
    particles: the one-launch solve keeps one block, then two, to a
    work-group, then lets each take a range (of two scenes, in a batch)."""
    counts = 64
    descs, parts = [], []
    for k in range(scenes):
        r = np.random.default_rng(7 + k)
        d, _, _, _ = M.scene_generate("two_balls", counts, 0)
        d.cg_max_iterations = 200
        x = r.uniform(0.15, 0.85, (n, 3)).astype(np.float32)
        x = np.concatenate([x, x + r.uniform(-0.5, 0.5, x.shape).astype(np.float32) / counts]).astype(np.float32)
        v = ((x - 0.5) @ r.uniform(-1.0, 1.0, (3, 3)) + 0.5).astype(np.float32)
        descs.append(d)
        parts.append((x, v, np.full(len(x), 400.0 / counts ** 3 / 8, np.float32)))
    dt = 0.5 * float(descs[0].max_dt)
    b = M.Batch(descs, [2 * n] * scenes)
    for k, (x, v, m) in enumerate(parts):
        b.upload(k, x, v, m)
    b.initialize()
    b.use_graph(graph)
    b.substep(dt)
    assert sum(b.stats(k)["active_blocks"] for k in range(scenes)) == blocks
    b.substep(dt)
    for k, (x, v, m) in enumerate(parts):
        o = O.Oracle(descs[k], 8, 4, O.DOT_FP64 | O.SVD_FP64)
        o.set_particles(x, v, m)
        o.initialize()
        for _ in range(2):
            o.advance_step(dt)
        got, want = b.download(k), o.particles()
        assert np.array_equal(got["ids"], want["ids"])
        for f in ("x", "v", "F", "Jp"):
            assert rel(got[f], want[f]) < 1e-5, (k, f)
    b.close()


def scattered(dim, counts, n, seed, lo=0.15, hi=0.85):
    r = np.random.default_rng(seed)
    name = "disk2d" if dim == 2 else "two_balls"
    d, _, _, _ = M.scene_generate(name, counts, 0)
    d.cg_max_iterations = 30
    x = r.uniform(lo, hi, (n, dim)).astype(np.float32)
    v = ((x - 0.5) @ r.uniform(-1.0, 1.0, (dim, dim)) + 0.5).astype(np.float32)
    return d, x, v, np.full(n, 400.0 / counts ** dim / 8, np.float32)


# (dimension, cells, particles and part of the domain of each scene, graph): a few
# groups of blocks; more than 192 of them; more than the launch has
# work-groups; the same in 2D; scenes that share groups, one of them with few blocks
@pytest.mark.parametrize("dim,counts,scenes,graph", [
    (3, 64, [(66000, 0.4, 0.6)], False),
    (3, 128, [(66000, 0.35, 0.65)], True),
    (3, 128, [(66000, 0.2, 0.8)], False),
    (2, 512, [(66000, 0.05, 0.95)], False),
    (3, 64, [(500, 0.4, 0.6), (66000, 0.2, 0.8), (300, 0.45, 0.5)], False),
    (3, 64, [(500, 0.4, 0.6), (66000, 0.2, 0.8), (300, 0.45, 0.5)], True),
])
def test_node_pass_work_groups(dim, counts, scenes, graph):
    """The node pass of launched solves (over 65,536 particles): one substep
    against the oracle, and two bit for bit the same with a wait limit of zero,
    where those that happen to run share the groups."""
    parts = [scattered(dim, counts, n, 40 + k, lo, hi) for k, (n, lo, hi) in enumerate(scenes)]
    dt = 0.5 * float(parts[0][0].max_dt)
    got = []
    for limit in (None, 0):
        b = M.Batch([q[0] for q in parts], [3 * len(q[1]) for q in parts])  # (a block per 16 places)
        if limit is not None:
            b.set_wait_limit(limit)
        for k, (_, x, v, m) in enumerate(parts):
            b.upload(k, x, v, m)
        b.initialize()
        b.use_graph(graph)
        b.substep(dt)
        once = [b.download(k) for k in range(len(parts))]
        b.substep(dt)
        got.append([(b.download(k), b.stats(k)) for k in range(len(parts))])
        b.close()
    for k, (d, x, v, m) in enumerate(parts):
        (a, sa), (c, sc) = got[0][k], got[1][k]
        assert sa["cg_iterations"] == sc["cg_iterations"] and sa["cg_multiplies"] == sc["cg_multiplies"]
        for f in ("x", "v", "F", "Jp", "ids"):
            assert np.array_equal(a[f], c[f]), f
        o = O.Oracle(d, 8, 4, O.DOT_FP64 | O.SVD_FP64)
        o.set_particles(x, v, m)
        o.initialize()
        o.advance_step(dt)
        want = o.particles()
        assert np.array_equal(once[k]["ids"], want["ids"])
        for f in ("x", "v", "F", "Jp"):
            assert rel(once[k][f], want[f]) < 1e-5, (k, f)


def test_solves_of_two_handles_at_once():
    """Work-groups of two launches that each exchange sums share the device:
    handles driven from two threads end as they do one after the other."""
    parts = [scattered(3, 64, 66000, 50, 0.2, 0.8), scattered(3, 64, 66000, 51, 0.3, 0.7), scattered(3, 32, 4000, 52, 0.3, 0.7)]
    dt = 0.5 * float(parts[0][0].max_dt)

    def handle(q):
        d, x, v, m = q
        s = M.Scene(d, 3 * len(m))
        s.upload(x, v, m)
        s.initialize()
        return s

    def drive(s):
        for _ in range(4):
            s.substep(dt)

    want = []
    for q in parts:
        s = handle(q)
        drive(s)
        want.append(s.download())
        s.close()
    scenes = [handle(q) for q in parts]
    threads = [threading.Thread(target=drive, args=(s,)) for s in scenes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s, w in zip(scenes, want):
        got = s.download()
        s.close()
        for f in ("x", "v", "F", "Jp", "ids"):
            assert np.array_equal(got[f], w[f]), f


# cells an axis around which the binning's scan changes form: up to 4,096 and
# 8,192 slots (3D 52 and 68 cells; 2D 496 has 4,225), alone and in a batch
@pytest.mark.parametrize("dim,counts", [(3, 48), (3, 52), (3, 56), (3, 68), (3, 72), (3, 88), (3, 92), (2, 496), (2, 504), (2, 1000)])
def test_scan_by_number_of_slots(dim, counts):
    parts = [scattered(dim, counts, n, 60 + n, 0.02, 0.98) for n in (400, 3)]
    dt = 0.5 * float(parts[0][0].max_dt)
    b = M.Batch([q[0] for q in parts[:1]], [2000])
    two = M.Batch([q[0] for q in parts], [2000, 100])
    for h, m in ((b, 1), (two, 2)):
        for k in range(m):
            h.upload(k, *parts[k][1:])
        h.initialize()
        h.substep(dt)
    for k, (d, x, v, m) in enumerate(parts):
        o = O.Oracle(d, 8, 4, O.DOT_FP64 | O.SVD_FP64)
        o.set_particles(x, v, m)
        o.initialize()
        o.advance_step(dt)
        want = o.particles()
        for got in [two.download(k)] + ([b.download(0)] if k == 0 else []):
            assert np.array_equal(got["ids"], want["ids"])
            for f in ("x", "v", "F", "Jp"):
                assert rel(got[f], want[f]) < 1e-5, (k, f)
    b.close()
    two.close()


@pytest.mark.parametrize("dim,counts,n", [(3, 64, 130), (2, 256, 250), (3, 64, 8)])
def test_one_block_to_a_work_group_repeats(dim, counts, n):
    """The one-launch solve with a block to a work-group, where waves poll for
    their neighbours' r ahead of their scene's sum: launched and replayed over
    many iterations, the same bit for bit whatever the work-groups' timing."""
    d, x, v, m = scattered(dim, counts, n, 70)
    dt = 0.5 * float(d.max_dt)
    runs = []
    for graph in (False, True, True):
        s = M.Scene(d, 2 * n)
        s.upload(x, v, m)
        s.initialize()
        s.use_graph(graph)
        runs.append(s)
    iterations = 0
    for step in range(40):
        stats = [s.substep(dt, stats=True) for s in runs]
        iterations += stats[0]["cg_iterations"]
        assert stats[0]["active_blocks"] <= 512
        got = [s.download() for s in runs]
        for k in (1, 2):
            assert stats[k] == stats[0], step
            for f in ("x", "v", "F", "Jp", "ids"):
                assert np.array_equal(got[k][f], got[0][f]), (step, k, f)
    assert iterations > 200
    for s in runs:
        s.close()


@contextlib.contextmanager
def busy_device():
    """Another handle's substeps, of work-groups of thousands of particles each,
    run meanwhile."""
    d, x, v, m = M.scene_generate("two_balls", 96, 5, 1_000_000)
    busy = M.Scene(d, len(m))
    busy.upload(x, v, m)
    busy.initialize()
    stop = threading.Event()

    def hold():
        while not stop.is_set():
            busy.substep(0.1 * float(d.max_dt))

    other = threading.Thread(target=hold)
    other.start()
    try:
        yield
    finally:
        stop.set()
        other.join()
        busy.close()


@pytest.mark.parametrize("counts,scenes", [(128, [(66000, 0.35, 0.65)]), (64, [(500, 0.4, 0.6), (66000, 0.2, 0.8), (300, 0.45, 0.5)])])
def test_node_pass_on_a_busy_device(counts, scenes):
    """Another handle's work-groups, of thousands of particles each, hold the
    device for longer than the wait limits, so that work-groups of a node pass
    start when those that found a place have shared the groups and finished.
    Particles, statistics and the solve's own arrays are those of an idle device
    bit for bit."""
    parts = [scattered(3, counts, n, 40 + k, lo, hi) for k, (n, lo, hi) in enumerate(scenes)]
    dt = 0.5 * float(parts[0][0].max_dt)

    def drive(limit):
        if len(parts) == 1:
            h = M.Scene(parts[0][0], 3 * len(parts[0][1]))
            h.upload(*parts[0][1:])
        else:
            h = M.Batch([q[0] for q in parts], [3 * len(q[1]) for q in parts])
            for k, q in enumerate(parts):
                h.upload(k, *q[1:])
        if limit is not None:
            h.set_wait_limit(limit)
        h.initialize()
        h.use_graph(True)
        out = []
        for _ in range(4):
            h.substep(dt)
            if len(parts) == 1:
                out.append([{**h.download(), "stats": h.stats(), "r": h.read_grid(M.CH_CG_R), "s": h.read_grid(M.CH_CG_S),
                             "q": h.read_grid(M.CH_CG_Q)}])
            else:
                out.append([{**h.download(k), "stats": h.stats(k)} for k in range(len(parts))])
        h.close()
        return out

    want = drive(None)
    with busy_device():
        got = [drive(None), drive(0)]
    for run, steps in enumerate(got):
        for step, (a, b) in enumerate(zip(steps, want)):
            for k in range(len(parts)):
                assert a[k]["stats"] == b[k]["stats"], (run, step, k)
                for f in a[k]:
                    if f != "stats":
                        assert np.array_equal(a[k][f], b[k][f]), (run, step, k, f)


def solved(parts, graph, limit, steps):
    """Particles, statistics and (one scene) the solve's arrays after each
    substep, and the active blocks of all scenes after the first."""
    dt = 0.5 * float(parts[0][0].max_dt)
    if len(parts) == 1:
        h = M.Scene(parts[0][0], 2 * len(parts[0][1]))
        h.upload(*parts[0][1:])
    else:
        h = M.Batch([q[0] for q in parts], [2 * len(q[1]) for q in parts])
        for k, q in enumerate(parts):
            h.upload(k, *q[1:])
    if limit is not None:
        h.set_wait_limit(limit)
    h.initialize()
    h.use_graph(graph)
    out = []
    for _ in range(steps):
        h.substep(dt)
        if len(parts) == 1:
            out.append([{**h.download(), "stats": h.stats(), "r": h.read_grid(M.CH_CG_R), "s": h.read_grid(M.CH_CG_S),
                         "q": h.read_grid(M.CH_CG_Q)}])
        else:
            out.append([{**h.download(k), "stats": h.stats(k)} for k in range(len(parts))])
    h.close()
    return out, sum(o["stats"]["active_blocks"] for o in out[0])


def assert_same_bits(got, want, where):
    for f in set(got) & set(want):
        if f == "stats":
            assert got[f] == want[f], where
        else:
            assert np.array_equal(got[f], want[f]), (where, f)


# (dimension, cells, particles of each scene, blocks): one scene with a block to a
# work-group and with two, two and three scenes with two, and ranges of blocks
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("dim,counts,sizes,blocks", [
    (3, 64, [130], (1, 512)), (2, 256, [250], (1, 512)), (3, 64, [250], (513, 1024)), (3, 64, [130, 130], (513, 1024)),
    (2, 256, [300, 3, 250], (513, 1024)), (3, 64, [250, 5, 300], (1025, 4096))])
def test_one_launch_solve_with_few_work_groups(dim, counts, sizes, blocks, graph):
    """Beside another handle's long work-groups, and with a wait limit of zero, the
    solve's door closes on those that happen to run: they share the blocks and
    end with the same bits as all of them on an idle device."""
    parts = [scattered(dim, counts, n, 80 + k) for k, n in enumerate(sizes)]
    want, nb = solved(parts, graph, None, 6)
    assert blocks[0] <= nb <= blocks[1]
    with busy_device():
        runs = [solved(parts, graph, limit, 6)[0] for limit in (0, None)]
    for got in runs:
        for step in range(6):
            assert got[step][0]["stats"]["cg_iterations"] > 3
            for k in range(len(parts)):
                assert_same_bits(got[step][k], want[step][k], (step, k))


@pytest.mark.parametrize("n,lo,hi,many", [(300, 0.3, 0.7, False), (900, 0.1, 0.9, True), (900, 0.28, 0.72, None)])
def test_form_of_the_solve_by_blocks(n, lo, hi, many):
    """Few particles over more blocks than the one-launch solve keeps resident
    take the launched kernels: from the start, or (None) from the third substep
    after the particles have spread over so many; replays take the same
    kernels as launched substeps, bit for bit, across the change."""
    d, x, v, m = scattered(3, 64, n, 90, lo, hi)
    if many is None:
        v = (60 * (x - 0.5)).astype(np.float32)
    runs = []
    for graph in (False, True):
        s = M.Scene(d, 20 * n)
        s.upload(x, v, m)
        s.initialize()
        s.use_graph(graph)
        runs.append(s)
    runs[0].enable_timing()
    blocks, launched, nodes = [], [], 0
    for step in range(16):
        st = [s.substep(1e-3, stats=True) for s in runs]
        assert st[0] == st[1], step
        blocks.append(st[0]["active_blocks"])
        now = runs[0].kernel_times()["cg_node"][1]
        launched.append(now > nodes)
        nodes = now
        a, b = (s.download() for s in runs)
        for f in ("x", "v", "F", "Jp", "ids"):
            assert np.array_equal(a[f], b[f]), (step, f)
    if many is None:
        assert min(blocks) <= 1024 < max(blocks)
    assert launched[2:] == [k > 1024 for k in blocks[:-2]]
    assert many is None or launched == [many] * 16
    for s in runs:
        s.close()


# (dimension, cells, particles, blocks): either side of the number of blocks up to
# which P2G takes a work-group per block
@pytest.mark.parametrize("dim,counts,n,blocks", [(3, 64, 730, (1500, 1536)), (3, 64, 744, (1537, 1560)), (2, 512, 1400, (1400, 1536)),
                                                 (2, 512, 1700, (1537, 1800))])
def test_p2g_by_number_of_blocks(dim, counts, n, blocks):
    d, x, v, m = scattered(dim, counts, n, 95, 0.1, 0.9)
    s = M.Scene(d, 20 * n)
    s.upload(x, v, m)
    s.initialize()
    assert blocks[0] <= s.stats()["active_blocks"] <= blocks[1]
    mass, vel = s.read_grid(M.CH_MASS), s.read_grid(M.CH_VELOCITY)  # of the initialisation
    s.close()
    o = O.Oracle(d, 8, 4, O.DOT_FP64 | O.SVD_FP64)
    o.set_particles(x, v, m)
    o.initialize()
    want = o.grid(M.CH_MASS)
    assert rel(mass, want) < 1e-5
    assert rel(mass[..., None] * vel, want[..., None] * o.grid(M.CH_VELOCITY)) < 1e-5
