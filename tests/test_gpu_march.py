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
