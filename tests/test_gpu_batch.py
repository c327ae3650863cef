"""Batched form: many uneven ray lists over several resident datasets traced
pass by pass by the persistent kernel give, list by list, the results of the
per-list loop (gxy_process_raylist / gxy_sample_raylist), and those of the
oracle; every launch configuration and the graph-captured run give the same
results; lists added while others are in flight (continuous form) get the
results they get alone."""
import ctypes as C

import numpy as np
import pytest

from batch_scenes import dataset_descs
from galaxy_amd import abi, scenes, workloads

pytestmark = pytest.mark.gpu
f32 = np.float32

SIZES = [1, 63, 64, 65, 200, 777, 1000, 2048, 3001, 5, 4096, 129]


@pytest.fixture(scope="module")
def datasets(hip):
    descs = dataset_descs()
    return descs, [scenes.build_scene(hip, sc) for sc in descs]


def lights_struct(keep):
    return scenes.make_lighting(workloads.batch_lighting(), keep)


def plain_list(L, built, lights, n, seed, ds_kind):
    """The per-list loop on the same rays: (fb, FrameStats)."""
    from galaxy_amd import batch as gb
    from galaxy_amd import lib as glib
    d = gb.random_rays(n, seed, width=n)
    fb = glib.DeviceArray(16 * n).zero()
    st = abi.FrameStats()
    nb = np.full(6, -1, np.int32)
    glib.check(L.gxy_process_raylist(C.byref(built.vis), C.byref(lights), n, C.byref(d.ispc), nb.ctypes.data, 0.001,
                                      1 << 30, fb.ptr, n, 1, C.byref(st)), "process_raylist")
    return fb.to_host(f32).reshape(-1, 4), st


def make_batch(built, lights, plan, chunk=256):
    from galaxy_amd import batch as gb
    B = gb.Batch(chunk)
    ids = [B.add_dataset(b) for b in built]
    B.set_lighting(lights)
    out = []
    for n, ds, seed in plan:
        d = gb.random_rays(n, seed, width=n)
        l, fb = B.add_render_list(ids[ds], d, n, 1)
        B.set_seed(l, seed)
        out.append((l, fb))
    return B, out


def plan_of(sizes, nds, seed0=100):
    return [(n, k % nds, seed0 + k) for k, n in enumerate(sizes)]


def test_batch_equals_per_list_loop(datasets, hip):
    from galaxy_amd import lib as glib
    L = glib.lib()
    descs, built = datasets
    keep = []
    lights = lights_struct(keep)
    plan = plan_of(SIZES, len(built))
    B, lists = make_batch(built, lights, plan)
    st = B.run(0)
    assert st.overflow == 0
    tot = dict(rays=0, samples=0, spawned=0, terminated=0, dropped=0, kept=0)
    for (n, ds, seed), (l, fb) in zip(plan, lists):
        ref, s = plain_list(L, built[ds], lights, n, seed, ds)
        got = fb.to_host(f32).reshape(-1, 4)
        # per-ray results are identical; only the order of float additions into a pixel may differ
        assert np.abs(got - ref).max() <= 1e-5, (n, ds)
        tot["rays"] += s.ray_passes
        tot["samples"] += s.samples
        tot["spawned"] += s.secondary_rays
        tot["terminated"] += s.terminated
        tot["dropped"] += s.dropped
        tot["kept"] += s.kept
    got = {k: getattr(st, k) for k in tot}
    assert got == tot, (got, tot)
    assert st.spawned > 1000 and st.samples > 100000


def test_graph_run_and_every_configuration_agree(datasets, hip):
    from galaxy_amd import batch as gb
    descs, built = datasets
    keep = []
    lights = lights_struct(keep)
    plan = plan_of(SIZES, len(built), 300)
    B, lists = make_batch(built, lights, plan)
    st0 = B.run(0)
    ref = [fb.to_host(f32) for _, fb in lists]
    depth = 0
    for b in built:
        if b.vis.model:
            nodes, leaves, dp, sah = C.c_int(), C.c_int(), C.c_int(), C.c_float()
            B.L.gxy_model_bvh_stats(b.vis.model, C.byref(nodes), C.byref(leaves), C.byref(dp), C.byref(sah))
            depth = max(depth, dp.value)
    runs = 0
    for cfg in gb.DEFAULT_CANDIDATES + [(64, 0, 0, 1), (1024, 0, 0, 2)]:
        if cfg[1] and depth + 2 > cfg[1]:
            continue
        B.set_config(*cfg)
        for gp in (0, 2):
            st = B.run(gp)
            assert st.overflow == 0
            for k in ("rays", "samples", "spawned", "terminated", "dropped", "kept"):
                assert getattr(st, k) == getattr(st0, k), (cfg, gp, k)
            for (l, fb), r in zip(lists, ref):
                assert np.abs(fb.to_host(f32) - r).max() <= 1e-5, (cfg, gp, l)
            runs += 1
    assert runs >= 8
    # graph replays after eager work in between give the same results again
    for _ in range(3):
        st = B.run(2)
        assert st.rays == st0.rays
        for (l, fb), r in zip(lists, ref):
            assert np.abs(fb.to_host(f32) - r).max() <= 1e-5


def test_batch_against_oracle(datasets, hip, oracle):
    """A few lists checked straight against the CPU restatement."""
    from galaxy_amd import batch as gb
    descs, built = datasets
    keep = []
    lights = lights_struct(keep)
    plan = plan_of([3000, 2500, 4000, 1500], len(built), 700)
    B, lists = make_batch(built, lights, plan)
    B.run(0)
    nb = np.full(6, -1, np.int32)
    for (n, ds, seed), (l, fb) in zip(plan, lists):
        hr = gb.random_rays(n, seed, width=n).download()
        Bo = scenes.build_scene(oracle, descs[ds])
        fbo = np.zeros(4 * n, f32)
        so = abi.FrameStats()
        oracle.L.oracle_process_raylist(C.byref(Bo.vis), C.byref(lights), hr.n,
                                        C.byref(hr.ispc), nb.ctypes.data, 0.001, 1 << 30, fbo.ctypes.data, n, 1,
                                        C.byref(so))
        got = fb.to_host(f32)
        assert np.abs(got - fbo).max() <= 1e-4, (n, ds)
        assert np.sqrt(np.mean((got - fbo) ** 2)) <= 1e-5


def test_sample_lists_equal_sampler_loop(datasets, hip):
    from galaxy_amd import batch as gb
    from galaxy_amd import lib as glib
    L = glib.lib()
    descs, built = datasets
    B = gb.Batch(128)
    ids = [B.add_dataset(b) for b in built]
    keep = []
    B.set_lighting(lights_struct(keep))
    cap = 400000
    runs = []
    for k, n in enumerate([5000, 777, 20000]):
        d = gb.random_rays(n, 900 + k, width=n)
        l, xyz, cnt = B.add_sample_list(ids[k % 2], d, cap)
        B.set_seed(l, 900 + k)
        runs.append((n, k % 2, 900 + k, xyz, cnt))
    # a render list in the same batch
    d = gb.random_rays(3000, 950, width=3000)
    lr, fbr = B.add_render_list(ids[3], d, 3000, 1)
    B.set_seed(lr, 950)
    st = B.run(0)
    # sampler rays follow all their crossings within a pass; the render list needs its shadow/AO pass
    assert st.passes == 2
    for n, ds, seed, xyz, cnt in runs:
        c = int(cnt.to_host(np.int32, 1)[0])
        d = gb.random_rays(n, seed, width=n)
        xr = glib.DeviceArray(cap * 12)
        cr = C.c_int()
        fs = abi.FrameStats()
        glib.check(L.gxy_sample_raylist(C.byref(built[ds].vis), n, C.byref(d.ispc), 1 << 30, xr.ptr, cap,
                                        C.byref(cr), C.byref(fs)))
        assert c == cr.value > n // 4
        a = xyz.to_host(f32, 3 * c).reshape(-1, 3)
        b = xr.to_host(f32, 3 * c).reshape(-1, 3)
        # the same particles; their order across passes and lists differs
        a = a[np.lexsort(a.T)]
        b = b[np.lexsort(b.T)]
        assert np.array_equal(a, b)


@pytest.mark.parametrize("step_rays", [0, 1500])
def test_continuous_batching_alone_equals_mix(datasets, hip, step_rays):
    """Lists added while others are in flight, with passes run one at a time,
    get the results they get in a batch of their own; with a step budget the
    primary rays of the lists join over several steps, fewest left first."""
    from galaxy_amd import batch as gb
    descs, built = datasets
    keep = []
    lights = lights_struct(keep)
    plan = plan_of([4000, 1500, 64, 3000, 999, 2500, 10, 4096], len(built), 1200)
    alone = []
    for p in plan:
        B1, ls = make_batch(built, lights, [p])
        B1.run(0)
        alone.append(ls[0][1].to_host(f32))
        B1.destroy()
    B = gb.Batch(256)
    B.set_step_rays(step_rays)
    assert B.L.gxy_batch_get_step_rays(B.h) == step_rays
    ids = [B.add_dataset(b) for b in built]
    B.set_lighting(lights)
    fbs = {}
    pending_plan = list(enumerate(plan))
    queued = []
    steps = 0
    done = set()
    started = {}
    while len(done) < len(plan):
        # admit up to two new lists per step
        for _ in range(2):
            if pending_plan:
                k, (n, ds, seed) = pending_plan.pop(0)
                d = gb.random_rays(n, seed, width=n)
                l, fb = B.add_render_list(ids[ds], d, n, 1)
                fbs[k] = fb
                started[k] = l
        queued.append(B.step())
        steps += 1
        pend = B.pending(len(B.lists) + 8)
        assert queued[-1] == pend.sum()
        for k, l in list(started.items()):
            if pend[l] == 0:
                done.add(k)
                del started[k]
                B.remove_list(l)
        assert steps < 100
    for k in range(len(plan)):
        assert np.abs(fbs[k].to_host(f32) - alone[k]).max() <= 1e-5, k
    if step_rays:
        # 16169 primary rays, at most 1500 + 255 (a whole last chunk) per step
        assert steps >= 9


def test_bricked_volume_datasets_give_the_same_results(datasets, hip):
    from galaxy_amd import lib as glib
    L = glib.lib()
    descs, built = datasets
    keep = []
    lights = lights_struct(keep)
    plan = plan_of(SIZES, len(built), 1500)
    B, lists = make_batch(built, lights, plan)
    st0 = B.run(0)
    ref = [fb.to_host(f32) for _, fb in lists]
    vols = [b.handles[0] for b, d in zip(built, descs) if d.volume_vis]
    try:
        for lay in (8, 4):
            for v in vols:
                glib.check(L.gxy_volume_set_layout(v, lay))
            B.refresh_datasets(built)
            for gp in (0, 2):
                st = B.run(gp)
                for k in ("rays", "samples", "spawned", "terminated", "dropped", "kept"):
                    assert getattr(st, k) == getattr(st0, k), (lay, gp, k)
                for (l, fb), r in zip(lists, ref):
                    assert np.abs(fb.to_host(f32) - r).max() <= 1e-5, (lay, gp, l)
    finally:
        for v in vols:
            L.gxy_volume_set_layout(v, 0)


def test_sampler_segment_cap_gives_the_same_particles(datasets, hip):
    """A sampler ray that reaches the per-pass crossing cap continues in the
    next pass: particle sets, ray passes and samples do not depend on the cap."""
    from galaxy_amd import batch as gb
    descs, built = datasets
    ref = None
    for cap_seg in (4096, 3, 1):
        B = gb.Batch(128)
        B.set_max_segments(cap_seg)
        ids = [B.add_dataset(b) for b in built]
        keep = []
        B.set_lighting(lights_struct(keep))
        lists = []
        for k, n in enumerate([5000, 20000]):
            d = gb.random_rays(n, 1900 + k, width=n)
            l, xyz, cnt = B.add_sample_list(ids[k % 2], d, 400000)
            B.set_seed(l, 1900 + k)
            lists.append((xyz, cnt))
        st = B.run(2)
        got = []
        for xyz, cnt in lists:
            c = int(cnt.to_host(np.int32, 1)[0])
            a = xyz.to_host(f32, 3 * c).reshape(-1, 3)
            got.append(a[np.lexsort(a.T)])
        if ref is None:
            ref = (got, st.rays, st.samples, st.passes)     # the graph's two passes, the second empty
        else:
            assert st.rays == ref[1] and st.samples == ref[2], cap_seg
            assert st.passes >= ref[3], cap_seg
            if cap_seg == 1:
                assert st.passes > ref[3]
            for a, b in zip(got, ref[0]):
                assert np.array_equal(a, b), cap_seg
        B.destroy()


def test_batch_direct_lighting_equals_per_list_loop(datasets, hip):
    """The direct lighting model (gxy_set_reverse_lighting(0), taken by the
    batch when its lighting is set) gives the per-list loop's frames."""
    from galaxy_amd import lib as glib
    L = glib.lib()
    descs, built = datasets
    keep = []
    glib.check(L.gxy_set_reverse_lighting(0))
    try:
        lights = lights_struct(keep)
        plan = plan_of([64, 777, 3001, 129, 2048, 5], len(built), 500)
        B, lists = make_batch(built, lights, plan)
        st = B.run(0)
        assert st.overflow == 0
        for (n, ds, seed), (l, fb) in zip(plan, lists):
            ref, s = plain_list(L, built[ds], lights, n, seed, ds)
            assert np.abs(fb.to_host(f32).reshape(-1, 4) - ref).max() <= 1e-5, (n, ds)
    finally:
        glib.check(L.gxy_set_reverse_lighting(1))


def test_pending_counts_lists_added_after_a_step(datasets, hip):
    """Lists added after a step report their waiting rays only: the pass
    counters cover the lists of the last passes and no entry beyond them."""
    from galaxy_amd import batch as gb
    descs, built = datasets
    keep = []
    lights = lights_struct(keep)
    B, lists = make_batch(built, lights, plan_of([500, 700, 900], len(built), 700))
    B.step()
    extra = []
    for k, n in enumerate((1000, 3000, 50, 4096, 7)):
        d = gb.random_rays(n, 800 + k, width=n)
        l, fb = B.add_render_list(k % len(built), d, n, 1)
        extra.append((l, n))
    p = B.pending(3 + len(extra))
    assert all(0 <= v <= 50 * 900 for v in p[:3])
    assert [int(p[l]) for l, _ in extra] == [n for _, n in extra]


def test_stack_check_counts_the_levels_of_the_width_asked_for(hip):
    """Width 4 with 32 stack entries takes a tree of 28 4-wide levels (55 binary
    ones), which the 4-wide walk itself does not, and refuses 24 entries."""
    from batch_scenes import graded_scene, rays_at_triangles
    from galaxy_amd import batch as gb
    from galaxy_amd import lib as glib
    L = glib.lib()
    sc = graded_scene(4)
    built = scenes.build_scene(hip, sc)
    n, keep, images = 2000, [], []
    x = np.arange(n, dtype=np.int32)
    try:
        for width, stack in ((2, 0), (4, 0), (4, 32), (4, 24)):
            glib.check(L.gxy_set_bvh_width(width))
            B = gb.Batch(128)
            hr = rays_at_triangles(sc, n, 3)
            hr["x"] = x
            hr["y"] = 0 * x
            d = glib.DeviceRays.from_host(hr)
            l, fb = B.add_render_list(B.add_dataset(built), d, n, 1)
            B.set_lighting(lights_struct(keep))
            B.set_config(128, stack, 0, 2)
            if stack == 24:
                with pytest.raises(glib.GxyError, match="BVH depth 28 needs"):
                    B.run(0)
                continue
            st = B.run(0)
            assert st.spawned > 1000
            images.append(fb.to_host(f32))
    finally:
        glib.check(L.gxy_set_bvh_width(2))
    for im in images[1:]:
        assert np.abs(im - images[0]).max() <= 1e-5


def _field(edge, seed=5, colormap=None):
    from batch_scenes import smooth_volume
    x = np.linspace(0.0, 1.0, 8)
    rgb, op = workloads.VOLUME_RENDER_TF
    vv = scenes.VolumeVisDesc(smooth_volume(edge, seed), colormap=np.c_[x, rgb].astype(f32) if colormap is None else colormap,
                              opacitymap=np.c_[x, 4 * op].astype(f32), isovalues=np.array([0.5], f32), volume_render=True)
    return scenes.SceneDesc(volume_vis=[vv], local_box=workloads.UNIT_BOX, global_box=workloads.UNIT_BOX)


def _camera_list(w, h, dist=1.9, aov=40.0):
    from galaxy_amd import lib as glib
    hip = glib.HipBackend()
    cam = scenes.CameraDesc((0.5 + 0.6 * dist, 0.9, 0.5 + 0.7 * dist), (0.5, 0.5, 0.5), (0, 1, 0), aov, w, h)
    return hip.camera_rays(cam, workloads.UNIT_BOX, workloads.UNIT_BOX, 1).download()


# one lane per ray and four: by the volume (96^3 in bricks, 48^3 linear), by the
# distance of the rays (pixels of 0.5 and of 10 voxels, random rays), by kind (up to
# 320^3 and 128^3 children follow their own rule), and for lists of up to 16 rays
@pytest.mark.parametrize("edge,layout", [(40, 0), (97, 4), (64, 0), (136, 8), (136, 0)])
@pytest.mark.parametrize("split", [0, 1])
def test_lanes_per_ray_of_a_chunk_do_not_show(hip, edge, layout, split):
    from galaxy_amd import batch as gb
    from galaxy_amd import lib as glib
    L = glib.lib()
    built = scenes.build_scene(hip, _field(edge))
    if layout:
        glib.check(L.gxy_volume_set_layout(built.handles[0], layout))
    keep = []
    lights = lights_struct(keep)
    lists = [(_camera_list(w, h), w, h) for w, h in ((200, 150), (16, 12), (4, 4))]
    for n in (700, 257, 16, 1):
        r = gb.random_rays(n, 40 + n, width=n).download()
        lists.append((r, n, 1))
    odd = gb.random_rays(300, 9, width=300).download()          # every kind in one list, some rays odd
    odd["type"] = np.arange(300) % 3 + 1
    for f, k in (("tMax", 7), ("ox", 30), ("dx", 61)):
        odd[f][k::90] = np.inf
        odd[f][k + 1::90] = np.nan
    lists.append((odd, 300, 1))
    B = gb.Batch(128)
    ds = B.add_dataset(built)
    B.set_lighting(lights)
    B.set_config(128, 0, 0, 4, split)
    fbs = []
    for hr, w, h in lists:
        d = glib.DeviceRays.from_host(hr)
        fbs.append(B.add_render_list(ds, d, w, h)[1])
        keep.append(d)
    st = B.run(0)
    tot = dict(rays=0, samples=0, spawned=0, terminated=0, dropped=0, kept=0)
    nb = np.full(6, -1, np.int32)
    for (hr, w, h), fb in zip(lists, fbs):
        ref, s = glib.DeviceArray(16 * w * h).zero(), abi.FrameStats()
        d = glib.DeviceRays.from_host(hr)
        glib.check(L.gxy_process_raylist(C.byref(built.vis), C.byref(lights), hr.n, C.byref(d.ispc), nb.ctypes.data, 0.001,
                                         1 << 30, ref.ptr, w, h, C.byref(s)))
        a, b = fb.to_host(f32), ref.to_host(f32)
        assert np.array_equal(np.isfinite(a), np.isfinite(b))
        ok = np.isfinite(b)
        assert np.abs(a[ok] - b[ok]).max() <= 1e-5, (w, h)
        for k, f in (("rays", "ray_passes"), ("samples", "samples"), ("spawned", "secondary_rays"),
                     ("terminated", "terminated"), ("dropped", "dropped"), ("kept", "kept")):
            tot[k] += getattr(s, f)
    assert {k: getattr(st, k) for k in tot} == tot
    assert st.spawned > 1000


@pytest.mark.parametrize("edge", [40, 64])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_unbounded_tables_in_a_batch(hip, edge, bad):
    """A transfer function with an infinity or a NaN: one lane per ray."""
    from galaxy_amd import batch as gb
    from galaxy_amd import lib as glib
    cm = np.array([[0, 0.2, 0.3, 0.4], [0.8, 0.5, 0.6, 0.7], [1.0, bad, 0.1, 0.1]], f32)
    built = scenes.build_scene(hip, _field(edge, 6, cm))
    keep = []
    lights = lights_struct(keep)
    plan = plan_of([5, 900, 4000], 1, 50)
    B, lists = make_batch([built], lights, plan, 128)
    B.run(0)
    seen = 0
    for (n, ds, seed), (l, fb) in zip(plan, lists):
        ref, _ = plain_list(glib.lib(), built, lights, n, seed, ds)
        got = fb.to_host(f32).reshape(-1, 4)
        assert np.array_equal(np.isfinite(got), np.isfinite(ref))
        ok = np.isfinite(ref)
        seen += (~ok).sum()
        assert np.abs(got[ok] - ref[ok]).max() <= 1e-5
    assert seen > 10


@pytest.mark.parametrize("cap", [1, 63, 64, 1000])
def test_particles_past_the_array_are_counted_not_written(datasets, hip, cap):
    from galaxy_amd import batch as gb
    from galaxy_amd import lib as glib
    _, built = datasets
    keep, runs, n, guard = [], [], 5000, 256
    for c in (400000, cap):
        B = gb.Batch(128)
        B.set_lighting(lights_struct(keep))
        d = gb.random_rays(n, 900, width=n)
        xyz, cnt = glib.DeviceArray.from_host(np.full(3 * (c + guard), -7.0, f32)), glib.DeviceArray(4).zero()
        glib.check(B.L.gxy_batch_add_list(B.h, B.add_dataset(built[0]), abi.BATCH_SAMPLE, n, C.byref(d.ispc), None, 0, 0,
                                          xyz.ptr, c, cnt.ptr))
        B.run(0)
        runs.append((xyz.to_host(f32, 3 * (c + guard)).reshape(-1, 3), int(cnt.to_host(np.int32, 1)[0])))
    (every, total), (some, counted) = runs
    assert cap < total <= 400000 and counted == total
    every = {p.tobytes() for p in every[:total]}
    assert all(p.tobytes() in every for p in some[:cap])
    assert (some[cap:] == -7.0).all()
