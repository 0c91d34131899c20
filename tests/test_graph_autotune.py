"""Captured substeps and the launch-shape autotuner.

A replayed graph must give what the launched substep gives: the graph runs
the CG to the largest cap with finished solves returning at once, and the
same kernels on the same layout do the same arithmetic in the same order
(binning sorts every cell stably), so every substep matches bit for bit, CG
iteration counts included.  Each replay is checked against the launched run,
with downloads (and so synchronisations) between replays.  Launch shapes
regroup only the CG's FP64 partial sums (the FP32 bar of one substep chain,
1e-5 relative L2), and tuning leaves the particle state as it was.
"""
import numpy as np
import pytest

import non_ficks_diffusion_amd as M

pytestmark = pytest.mark.gpu

SCENES = [("two_balls", 24, 0, 0), ("blob", 32, 1001, 20000), ("slab", 40, 1002, 8000)]


def rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def make_batch(data):
    b = M.Batch([d for d, _, _, _ in data], [len(m) for _, _, _, m in data])
    for k, (_, x, v, m) in enumerate(data):
        b.upload(k, x, v, m)
    b.initialize()
    return b


def load():
    return [M.scene_generate(n, c, s, k) for n, c, s, k in SCENES]


def assert_same(got, ref, what):
    assert np.array_equal(got["ids"], ref["ids"]), what
    for f in ("x", "v", "F", "Jp"):
        assert rel(got[f], ref[f]) < 1e-5, (what, f, rel(got[f], ref[f]))


def assert_identical(got, ref, what):
    for f in ("ids", "x", "v", "F", "Jp", "mass", "volume"):
        assert np.array_equal(got[f], ref[f]), (what, f)


def test_batch_graph_replays_match_launched_substeps():
    data = load()
    eager, graph = make_batch(data), make_batch(data)
    graph.use_graph(True)
    dts = [[1e-3, 1e-3, 5e-4], [1e-3, 5e-4, 5e-4], [5e-4, 0.0, 1e-3], [1e-3, 1e-3, 1e-3], [5e-4, 5e-4, 0.0]]
    for step, dt in enumerate(dts):
        eager.substep(dt)
        graph.substep(dt)
        for k in range(len(data)):
            assert_identical(graph.download(k), eager.download(k), (step, k))
            se, sg = eager.stats(k), graph.stats(k)
            assert se["cg_iterations"] == sg["cg_iterations"], (step, k)
            assert se["active_blocks"] == sg["active_blocks"], (step, k)
    eager.close()
    graph.close()


def test_single_scene_graph_replays_match_launched_substeps():
    d, x, v, m = M.scene_generate("two_balls", 32, 0)
    runs = []
    for g in (False, True):
        s = M.Scene(d, len(m))
        s.upload(x, v, m)
        s.initialize()
        s.use_graph(g)
        runs.append(s)
    for step in range(4):
        for s in runs:
            s.substep(1e-3)
        assert_identical(runs[1].download(), runs[0].download(), step)
        assert runs[1].stats()["cg_iterations"] == runs[0].stats()["cg_iterations"], step
    for s in runs:
        s.close()


def test_graph_rejects_uncapped_cg():
    d, x, v, m = M.scene_generate("ref3d_test18", 20, 0)  # CG cap 10000
    s = M.Scene(d, len(m))
    with pytest.raises(M.MPMError):
        s.use_graph(True)
    s.close()


def test_autotune_keeps_particles_and_results():
    data = load()
    tuned, plain = make_batch(data), make_batch(data)
    dt = [1e-3, 1e-3, 1e-3]
    before = [tuned.download(k) for k in range(len(data))]
    cfg = tuned.autotune(dt)
    for k in range(len(data)):
        after = tuned.download(k)
        for f in ("x", "v", "F", "Jp", "volume"):
            assert np.array_equal(after[f], before[k][f]), (k, f)
    for key in ("block_groups", "node_groups", "particle_groups"):
        assert cfg[key] % 8 == 0 and cfg[key] >= 8
    assert tuned.launch_config()["block_groups"] == cfg["block_groups"]
    for _ in range(3):
        tuned.substep(dt)
        plain.substep(dt)
    for k in range(len(data)):
        assert_same(tuned.download(k), plain.download(k), k)
    # same size bucket: the cached result, no timing
    again = make_batch(data)
    cached = again.autotune(dt, cached=True)
    assert cached["from_cache"] == 1
    assert cached["block_groups"] == cfg["block_groups"]
    for b in (tuned, plain, again):
        b.close()


@pytest.mark.parametrize("operator_mode", [0, 1])
def test_launch_config_shapes_do_not_change_results(operator_mode):
    data = load()
    a, b = make_batch(data), make_batch(data)
    b.set_launch_config(64, 128, 16, operator_mode=operator_mode, operator_groups=40)
    b.use_graph(True)
    for _ in range(3):
        a.substep(1e-3)
        b.substep(1e-3)
    for k in range(len(data)):
        assert_same(b.download(k), a.download(k), k)
    with pytest.raises(M.MPMError):
        b.set_launch_config(100, 128, 16)  # not a multiple of 8
    with pytest.raises(M.MPMError):
        b.set_launch_config(64, 4096, 16)  # node work-groups above 2048
    with pytest.raises(M.MPMError):
        b.set_launch_config(64, 128, 16, operator_mode=2)
    a.close()
    b.close()


def test_single_scene_operator_modes_agree():
    """One wave per block (a lane runs its whole cell, scatter accumulated in
    registers) against four waves per block, on the single-scene path."""
    d, x, v, m = M.scene_generate("avalanche", 64, 0)
    runs = []
    for mode in (0, 1):
        s = M.Scene(d, len(m))
        s.upload(x, v, m)
        s.initialize()
        cfg = s.launch_config()
        s.set_launch_config(cfg["block_groups"], cfg["node_groups"], cfg["particle_groups"], operator_mode=mode,
                            operator_groups=cfg["operator_groups"] if mode == 0 else 256)
        for _ in range(3):
            s.substep(1e-3)
        runs.append(s)
    assert_same(runs[1].download(), runs[0].download(), "modes")
    for s in runs:
        s.close()


def host_rule_steps(d, time, target, vmax=0.0):
    """MPM_Driver::Advance_To_Target_Time's dt sequence in float32 arithmetic
    (MPM_Driver.cpp:55-80) for a constant max speed."""
    f = np.float32
    t, tgt, n = f(time), f(target), 0
    dx = f(1.0) / f(d.counts)
    while True:
        v = f(vmax)
        dt = f(d.cfl) * dx / (f(1e-2) if v < f(1e-2) else v)
        dt = dt if dt < f(d.max_dt) else f(d.max_dt)
        dt = dt if f(d.min_dt) < dt else f(d.min_dt)
        last = False
        if tgt - t < dt * f(1.001):
            dt, last = tgt - t, True
        elif tgt - t < f(2.0) * dt:
            dt = (tgt - t) * f(0.5)
        if not dt > 0:
            break
        t = f(t + dt)
        n += 1
        if last:
            break
    return float(t), n


def test_device_frame_loop_takes_the_host_rules_dts():
    """Captured substeps advance to a frame end with the dt rule on the
    device.  A scene at rest without gravity keeps max |V| = 0, so the dt
    sequence is fixed: the substep count and the end time equal the rule's
    in float32 arithmetic, including the end-of-frame halving."""
    d, x, v, m = M.scene_generate("two_balls", 24, 0)
    d.gravity[:] = (0.0, 0.0, 0.0)
    v = np.zeros_like(v)
    s = M.Scene(d, len(m))
    s.upload(x, v, m)
    s.initialize()
    s.use_graph(True)
    t = 0.0
    for frame in (1, 2, 3):
        target = float(np.float32(frame) / np.float32(24.0))
        t_exp, n_exp = host_rule_steps(d, t, target)
        t, n, _ = s.advance_to_time(t, target)
        assert n == n_exp and t == t_exp, (frame, n, n_exp, t, t_exp)
    assert s.max_particle_velocity() == 0.0
    s.close()


def test_device_frame_loop_matches_host_loop():
    """A batch advanced a frame by the device loop (captured substeps) and by
    the host loop (launched substeps): equal substep counts per scene, end
    times within float rounding, states to the bar of a substep chain."""
    data = load()
    host, dev = make_batch(data), make_batch(data)
    dev.use_graph(True)
    target = float(np.float32(1.0) / np.float32(24.0))
    th, nh = host.advance_to_time(0.0, target)
    td, nd = dev.advance_to_time(0.0, target)
    assert np.array_equal(nh, nd), (nh, nd)
    assert np.allclose(th, td, rtol=1e-6, atol=0)
    for k in range(len(data)):
        a, b = host.download(k), dev.download(k)
        assert np.array_equal(a["ids"], b["ids"])
        for f in ("x", "v", "F"):
            assert rel(b[f], a[f]) < 1e-4, (k, f, rel(b[f], a[f]))
    host.close()
    dev.close()


def test_copy_bandwidth_roof_is_plausible():
    # a streaming copy of 256 MiB: well above PCIe rates, below the 8 TB/s peak
    gbs = M.measure_copy_bandwidth(1 << 28, 5)
    print("copy GB/s", gbs)
    assert 500.0 < gbs < 8000.0


def test_stage_timing_leaves_the_state_as_it_was():
    d, x, v, m = M.scene_generate("two_balls", 24, 0)
    runs = []
    for timed in (False, True):
        s = M.Scene(d, len(m))
        s.upload(x, v, m)
        s.initialize()
        s.substep(1e-3)
        before = s.download()
        if timed:
            for stage in (M.STAGE_P2G, M.STAGE_G2P, M.STAGE_CONSTITUTIVE):
                assert s.time_stage(stage, 5) > 0.0
            after = s.download()
            for f in ("ids", "x", "v", "F", "Jp", "volume"):
                assert np.array_equal(after[f], before[f]), f
        # what MPM_Driver reads next: the max speed, the stats and a frame
        # advanced with the dt rule from that max speed
        vmax = s.max_particle_velocity()
        st = s.stats()
        s.substep(1e-3)
        after_step = s.download()
        t, n, _ = s.advance_to_time(0.0, 1.0 / 240.0)
        runs.append((vmax, st, after_step, n, t, s.download()))
        s.close()
    (v0, st0, a0, n0, t0, f0), (v1, st1, a1, n1, t1, f1) = runs
    assert v1 == v0, (v1, v0)
    for k in ("live_particles", "max_speed", "active_blocks"):
        assert st1[k] == st0[k], (k, st1[k], st0[k])
    assert_same(a1, a0, "substep after stage timing")
    assert n1 == n0 and abs(t1 - t0) <= 1e-6 * t0, (n1, n0, t1, t0)
    assert_same(f1, f0, "frame after stage timing")


def launched_cg_handle(n=66000, counts=64):
    """A scene above the size whose CG is one launch."""
    r = np.random.default_rng(11)
    d, _, _, _ = M.scene_generate("two_balls", counts, 0)
    d.cg_max_iterations = 30
    x = r.uniform(0.3, 0.7, (n, 3)).astype(np.float32)
    v = ((x - 0.5) @ r.uniform(-1.0, 1.0, (3, 3)) + 0.5).astype(np.float32)
    s = M.Scene(d, n)
    s.upload(x, v, np.full(n, 400.0 / counts ** 3 / 8, np.float32))
    s.initialize()
    return s, 0.3 * float(d.max_dt)


def test_counts_follow_the_blocks_until_they_are_chosen():
    s, dt = launched_cg_handle()
    blocks = s.stats()["active_blocks"]
    cfg = s.launch_config()
    for key in ("block_groups", "operator_groups"):
        assert blocks <= cfg[key] <= 1.25 * blocks + 72 and cfg[key] % 8 == 0, key
    # set as reported: still following
    s.set_launch_config(cfg["block_groups"], cfg["node_groups"], cfg["particle_groups"], operator_groups=cfg["operator_groups"])
    s.use_graph(True)
    s.substep(dt)
    s.use_graph(False)
    s.substep(dt)
    assert s.launch_config()["block_groups"] <= 1.25 * s.stats()["active_blocks"] + 72
    # chosen: as chosen
    s.set_launch_config(4096, cfg["node_groups"], cfg["particle_groups"], operator_groups=40)
    s.substep(dt)
    got = s.launch_config()
    assert got["block_groups"] == 4096 and got["operator_groups"] == 40
    s.close()


def test_autotune_times_the_operator_where_it_is_launched():
    s, dt = launched_cg_handle()
    cfg = s.autotune(dt)
    assert cfg["operator_ms"] > 0
    got = s.launch_config()
    for key in ("block_groups", "node_groups", "particle_groups", "operator_groups"):
        assert got[key] == cfg[key], key
    s.close()
    d, x, v, m = M.scene_generate("two_balls", 32, 0)
    s = M.Scene(d, len(m))
    s.upload(x, v, m)
    s.initialize()
    cfg = s.autotune(dt)  # its CG is one launch
    assert cfg["operator_ms"] == 0 and cfg["block_ms"] > 0
    s.close()


@pytest.mark.parametrize("graph", [False, True])
def test_launched_operator_with_fewer_groups_than_blocks(graph):
    """A launched CG whose operator takes several blocks to a work-group."""
    runs = []
    for groups in (None, 24):
        s, dt = launched_cg_handle()
        if groups:
            cfg = s.launch_config()
            s.set_launch_config(groups, 64, cfg["particle_groups"], operator_groups=groups)
            assert groups < s.stats()["active_blocks"] // 8
        s.use_graph(graph)
        for _ in range(3):
            s.substep(dt)
        runs.append(s)
    assert_identical(runs[1].download(), runs[0].download(), groups)
    for s in runs:
        s.close()
