"""Volume marches with several lanes per ray against the one-ray-per-lane march:
list sizes around the lane-group rules, volumes from a few voxels up, rays that
enter, miss, start inside, end at once or step past the exit at the first step."""
import ctypes as C

import numpy as np
import pytest

from galaxy_amd import abi, scenes, workloads

pytestmark = pytest.mark.gpu
f32 = np.float32


def _volume(edge, seed, rate=0.5):
    from batch_scenes import smooth_volume
    vol = smooth_volume(edge, seed)
    vol.sampling_rate = rate
    x = np.linspace(0.0, 1.0, 8)
    rgb, op = workloads.VOLUME_RENDER_TF
    vv = scenes.VolumeVisDesc(vol, colormap=np.c_[x, rgb].astype(f32), opacitymap=np.c_[x, 4 * op].astype(f32),
                              isovalues=np.array([0.5, 0.7], f32), volume_render=True)
    return scenes.SceneDesc(volume_vis=[vv], local_box=workloads.UNIT_BOX, global_box=workloads.UNIT_BOX)


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    o = rng.uniform(-0.5, 1.5, (n, 3))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    t0, tm = np.zeros(n), np.full(n, 1e30)
    k = np.arange(n)
    d[k % 11 == 0] = np.eye(3)[rng.integers(3, size=(k % 11 == 0).sum())]
    o[k % 7 == 0] = rng.uniform(0, 1, ((k % 7 == 0).sum(), 3))      # from inside
    tm[k % 13 == 0] = rng.uniform(0.0, 0.4, (k % 13 == 0).sum())    # end early
    t0[k % 17 == 0] = rng.uniform(0.0, 3.0, (k % 17 == 0).sum())
    return abi.HostRays.from_arrays(o.astype(f32), d.astype(f32), t0.astype(f32), tm.astype(f32))


def _sample(hip, sc, layout, hr):
    from galaxy_amd import lib as glib
    L = glib.lib()
    B = scenes.build_scene(hip, sc)
    if layout:
        glib.check(L.gxy_volume_set_layout(B.handles[0], layout))
    d = glib.DeviceRays.from_host(hr)
    L.SamplerTraceRays_SamplerTraceRays(None, C.byref(B.vis), hr.n, C.byref(d.ispc))
    assert L.gxy_last_error() == b""
    glib.check(L.gxy_synchronize())
    return d.download()


# lists around the sixteen-lane rule (2^16) and the edges of a wave and a workgroup
@pytest.mark.parametrize("n", [1, 3, 63, 64, 257, 65536, 65537, 70001])
@pytest.mark.parametrize("edge,layout,rate", [(3, 0, 0.5), (9, 4, 0.5), (33, 8, 0.5), (33, 0, 0.3), (5, 0, 8.0)])
def test_sampler_lanes_take_the_one_ray_march(hip, n, edge, layout, rate):
    """Bit for bit the march of one ray per lane, which scenes of several volumes
    take: the second visualization's isovalue is never crossed."""
    sc = _volume(edge, 3, rate)
    hr = _rays(n, 5 + n)
    hr["term"] = -7
    g = _sample(hip, sc, layout, hr)
    two = _volume(edge, 3, rate)
    two.volume_vis = [two.volume_vis[0], scenes.VolumeVisDesc(two.volume_vis[0].volume, isovalues=np.array([99.0], f32))]
    r = _sample(hip, two, 0, hr)
    assert np.isin(g["term"], (abi.RAY_SURFACE, abi.RAY_BOUNDARY)).all()
    for f in ("t", "term"):
        assert np.array_equal(g[f].view(np.int32), r[f].view(np.int32)), f
    if n > 1000 and edge > 3 and rate < 1:
        assert 0.05 < np.mean(g["term"] == abi.RAY_SURFACE) < 0.95


# sixteen lanes per ray and, with rays that miss added, eight
@pytest.mark.parametrize("extra", [0, 65536])
def test_sampler_lanes_stop_at_the_step_limit(hip, extra):
    """Rays that leave the volume a few steps before, at and after the most steps
    that a march takes (2^20)."""
    limit = 1 << 20
    sc = _volume(3, 3, 2.0 / (1.06 * limit))             # (steps of half an edge times the rate)
    vol = sc.volume_vis[0].volume
    sc.volume_vis[0].isovalues = np.array([99.0], f32)   # never crossed
    step = f32(min(vol.spacing)) * f32(vol.sampling_rate)
    t = np.cumsum(np.full(limit + 40, step), dtype=f32)  # the positions, added up one by one
    assert t[-1] < 1.0
    n = 40
    o = np.full((n, 3), 0.3)
    o[:, 0] = 1.0 - t[limit - 12:limit + 28].astype(float)
    d = np.tile([1.0, 0.0, 0.0], (n, 1))
    o = np.concatenate([o, np.full((extra, 3), 9.0)])
    d = np.concatenate([d, np.tile([0.0, 0.0, 1.0], (extra, 1))])
    hr = abi.HostRays.from_arrays(o.astype(f32), d.astype(f32), np.zeros(n + extra, f32), np.full(n + extra, 1e30, f32))
    g = _sample(hip, sc, 0, hr)
    sc.volume_vis = [sc.volume_vis[0], scenes.VolumeVisDesc(vol, isovalues=np.array([99.0], f32))]
    r = _sample(hip, sc, 0, hr)
    assert len(np.unique(r["t"][:n])) > 10
    for f in ("t", "term"):
        assert np.array_equal(g[f].view(np.int32), r[f].view(np.int32)), (f, np.nonzero(g[f] != r[f])[0])


def _trace(hip, B, hr, kind):
    from galaxy_amd import lib as glib
    L = glib.lib()
    saved = [C.c_int() for _ in range(3)]
    L.gxy_get_trace_config(*[C.byref(x) for x in saved])
    glib.check(L.gxy_set_trace_config(kind, 256, 32))
    try:
        d = glib.DeviceRays.from_host(hr)
        assert hip.trace(B.vis, d) == ""
        return d.download()
    finally:
        L.gxy_set_trace_config(*[x.value for x in saved])


def _mixed_rays(n, seed):
    """Primary, shadow and AO rays with colours in hand, some of them odd."""
    hr = _rays(n, seed)
    rng = np.random.default_rng(seed)
    hr["type"] = rng.choice([abi.RAY_PRIMARY, abi.RAY_SHADOW, abi.RAY_AO], n)
    if n > 200:
        hr["type"][:128] = abi.RAY_PRIMARY
    for f in "rgb":
        hr[f] = rng.uniform(-0.3, 0.3, n)
    hr["o"] = rng.uniform(0, 0.5, n)
    for f, k in (("o", 5), ("r", 6), ("o", 7), ("g", 8)):
        for v, q in ((np.inf, 0), (-np.inf, 100), (np.nan, 200)):
            hr[f][k + q::1000] = v
    for f in ("sr", "sg", "sb", "so", "nx", "ny", "nz"):
        hr[f] = 0.25
    return hr


# 16 lanes up to 2^16 rays; at 16 march steps across the box 4096 rays per step
# (two lanes) and 5.6 K (one), at 64 steps 1 K (four)
@pytest.mark.parametrize("n,edge", [(1, 3), (15, 9), (257, 33), (65536, 9), (65537, 9), (90001, 9), (65537, 33)])
@pytest.mark.parametrize("layout,isos,slices,dvr", [(0, 1, 0, True), (4, 1, 0, True), (8, 0, 1, True), (0, 2, 2, True),
                                                    (4, 2, 0, False), (8, 1, 1, True), (0, 0, 1, False)])
def test_lanes_per_ray_give_the_one_lane_march(hip, n, edge, layout, isos, slices, dvr):
    from galaxy_amd import lib as glib
    sc = _volume(edge, 6)
    vv = sc.volume_vis[0]
    vv.isovalues, vv.volume_render = vv.isovalues[:isos], dvr
    vv.slices = np.array([[0, 0, 1, 0.4], [0.6, 0.8, 0, 0.7]], f32)[:slices]
    B = scenes.build_scene(hip, sc)
    if layout:
        glib.check(glib.lib().gxy_volume_set_layout(B.handles[0], layout))
    hr = _mixed_rays(n, 11 + n)
    a, b = _trace(hip, B, hr, 0), _trace(hip, B, hr, 16)
    for f in abi.FIELDS:
        x, y = a[f].view(np.int32), b[f].view(np.int32)
        if a[f].dtype == f32:      # (the bits of a NaN are not part of the result)
            x, y = np.where(np.isnan(a[f]), 0, x), np.where(np.isnan(b[f]), 0, y)
            assert np.array_equal(np.isnan(a[f]), np.isnan(b[f])), f
        assert np.array_equal(x, y), (f, np.nonzero(x != y)[0][:5])


def test_unbounded_tables_keep_the_one_lane_march(hip):
    """A table with an infinity or a NaN: weights of zero would spread it."""
    from galaxy_amd import lib as glib
    sc = _volume(17, 6)
    for bad in (np.inf, np.nan):
        vv = sc.volume_vis[0]
        vv.colormap = np.array([[0, 0.2, 0.3, 0.4], [0.8, 0.5, 0.6, 0.7], [1.0, bad, 0.1, 0.1]], f32)
        B = scenes.build_scene(hip, sc)
        hr = _mixed_rays(4000, 21)
        a, b = _trace(hip, B, hr, 0), _trace(hip, B, hr, 16)
        for f in abi.FIELDS:
            assert np.array_equal(a[f], b[f], equal_nan=a[f].dtype == f32), f


def _spoil(sc, seed):
    """NaN and infinite voxels here and there."""
    v = sc.volume_vis[0].volume
    data = np.array(v.voxels, f32)
    rng = np.random.default_rng(seed)
    at = rng.random(data.shape)
    data[at < 0.004], data[(at > 0.1) & (at < 0.104)], data[(at > 0.2) & (at < 0.204)] = np.nan, np.inf, -np.inf
    v.voxels = data
    return sc


@pytest.mark.parametrize("n,edge", [(4000, 17), (65537, 33), (65537, 9)])
def test_odd_voxels_take_the_one_lane_march(hip, n, edge):
    """A sample of NaN or infinity counts for nothing with several lanes per ray
    too, where it is a weight of 0 and not a branch."""
    sc = _spoil(_volume(edge, 6), 3)
    B = scenes.build_scene(hip, sc)
    hr = _mixed_rays(n, 31)
    a, b = _trace(hip, B, hr, 0), _trace(hip, B, hr, 16)
    for f in abi.FIELDS:
        assert np.array_equal(a[f], b[f], equal_nan=a[f].dtype == f32), f
    plain = _volume(edge, 6)                # a second volume without odd voxels: nothing in it crosses 99
    two = scenes.SceneDesc(volume_vis=[sc.volume_vis[0], scenes.VolumeVisDesc(plain.volume_vis[0].volume,
                                                                              isovalues=np.array([99.0], f32))],
                           local_box=workloads.UNIT_BOX, global_box=workloads.UNIT_BOX)
    g, r = _sample(hip, sc, 0, _rays(n, 7)), _sample(hip, two, 0, _rays(n, 7))
    for f in ("t", "term"):
        assert np.array_equal(g[f], r[f], equal_nan=True), f


@pytest.mark.parametrize("n", [1, 257, 65537, 90001])
@pytest.mark.parametrize("edge,layout", [(9, 0), (33, 4)])
def test_lanes_count_the_samples_of_the_one_lane_march(hip, n, edge, layout):
    from galaxy_amd import lib as glib
    L = glib.lib()
    sc = _volume(edge, 6)
    keep, stats = [], []
    lights = scenes.make_lighting(workloads.batch_lighting(), keep)
    nb = np.full(6, -1, np.int32)
    saved = [C.c_int() for _ in range(3)]
    L.gxy_get_trace_config(*[C.byref(x) for x in saved])
    B = scenes.build_scene(hip, sc)
    if layout:
        glib.check(L.gxy_volume_set_layout(B.handles[0], layout))
    hr = _rays(n, 3 + n)
    try:
        for kind in (0, 16):
            glib.check(L.gxy_set_trace_config(kind, 256, 32))
            d, fb, st = glib.DeviceRays.from_host(hr), glib.DeviceArray(16 * n).zero(), abi.FrameStats()
            glib.check(L.gxy_process_raylist(C.byref(B.vis), C.byref(lights), n, C.byref(d.ispc), nb.ctypes.data, 0.001,
                                             1 << 30, fb.ptr, n, 1, C.byref(st)))
            stats.append(st.as_dict())
    finally:
        L.gxy_set_trace_config(*[x.value for x in saved])
    assert stats[0] == stats[1] and (n == 1 or stats[0]["samples"] > n)
    # two volumes count two samples a step, but one at the crossings of the first
    counts = []
    two = scenes.SceneDesc(volume_vis=[sc.volume_vis[0], scenes.VolumeVisDesc(sc.volume_vis[0].volume,
                                                                              isovalues=np.array([99.0], f32))],
                           local_box=workloads.UNIT_BOX, global_box=workloads.UNIT_BOX)
    for s in (sc, two):
        B2 = scenes.build_scene(hip, s)
        if layout and s is sc:
            glib.check(L.gxy_volume_set_layout(B2.handles[0], layout))
        d, st, c = glib.DeviceRays.from_host(hr), abi.FrameStats(), C.c_int()
        xyz = glib.DeviceArray(12 * (40 * n + 100))
        glib.check(L.gxy_sample_raylist(C.byref(B2.vis), n, C.byref(d.ispc), 1 << 30, xyz.ptr, 40 * n + 100, C.byref(c),
                                        C.byref(st)))
        counts.append((st.samples, c.value))
    assert counts[0][1] == counts[1][1] and counts[1][0] == 2 * counts[0][0] - counts[0][1]
