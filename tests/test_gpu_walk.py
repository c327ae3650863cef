"""The 4-wide BVH walk against the binary one: the same hits, t, colours and
geometry / primitive IDs on every ray, the awkward ones included (axis-aligned
and denormal directions, origins on box faces, infinite and NaN fields, empty
intervals), over trees from one leaf to several thousand nodes."""
import ctypes as C

import numpy as np
import pytest

from galaxy_amd import abi, scenes, workloads

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module")
def hip():
    from galaxy_amd import lib as glib
    return glib.HipBackend()


def _scene(kind):
    rng = np.random.default_rng(3)
    box = ((-0.5,) * 3, (1.5,) * 3)
    sc = scenes.SceneDesc(local_box=box, global_box=box)
    if kind.startswith("tris"):
        # n triangles, axis-aligned ones (flat boxes) among them
        n = int(kind[4:])
        v = rng.uniform(0, 1, (n, 3, 3))
        v[::2] = v[::2, :1] + rng.uniform(-0.2, 0.2, (len(v[::2]), 3, 3))
        v[::3, :, 2] = v[::3, :1, 2]
        sc.meshes = [scenes.MeshDesc(v.reshape(-1, 3).astype(f32), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))]
    elif kind == "stacked":
        # many equal triangles: ties in t, a tree without spatial order
        v = np.tile(rng.uniform(0.2, 0.8, (4, 3, 3)), (300, 1, 1))
        sc.meshes = [scenes.MeshDesc(v.reshape(-1, 3).astype(f32), np.arange(3600, dtype=np.uint32).reshape(-1, 3))]
    elif kind == "blob_spheres":
        sc.meshes = [scenes.blob_mesh(20000, 5)]
        sc.spheres = [scenes.SpheresDesc(rng.uniform(0, 1, (3000, 3)).astype(f32), rng.uniform(0, 1, 3000).astype(f32),
                                         0.005, 0.03, 0.0, 1.0)]
    else:
        sc.pathlines = workloads.pathlines(8, 8, 200, 24, 2)[0].pathlines
    return sc


def _rays():
    rng = np.random.default_rng(8)
    n = 6000
    o = rng.uniform(-0.4, 1.4, (n, 3))
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    t0, tm = np.zeros(n), np.full(n, 1e30)
    for a in range(3):                       # axis-aligned, both ways, and nearly so
        k = slice(200 * a, 200 * a + 100)
        d[k] = 0.0
        d[k, a] = rng.choice([-1.0, 1.0], 100)
        k = slice(200 * a + 100, 200 * a + 200)
        d[k, a] = rng.choice([1e-30, -1e-30, 1e-40, -1e-44, -0.0, 1e-7], 100)
    o[600:700] = np.round(o[600:700])        # origins on the scene's faces and corners
    o[700:750] *= 1e4                        # far away, aimed back
    d[700:750] = (0.5 - o[700:750]) / np.linalg.norm(0.5 - o[700:750], axis=1, keepdims=True)
    tm[700:750] = 1e6
    t0[750:800] = 0.3
    tm[800:850] = 0.25
    t0[850:860], tm[850:860] = 0.5, 0.2      # an empty interval
    tm[860:870] = np.inf
    d[870:900] *= rng.choice([1e-8, 1e6, 1e-20], (30, 1))
    for k, v in ((900, np.nan), (910, np.inf), (920, -np.inf)):
        o[k:k + 3, 0] = v
        o[k + 3:k + 6, 2] = v
        d[k + 6:k + 8, 1] = v
        t0[k + 8] = v
        tm[k + 9] = v
    return abi.HostRays.from_arrays(o.astype(f32), d.astype(f32), t0.astype(f32), tm.astype(f32))


@pytest.mark.parametrize("kind", ["tris1", "tris2", "tris3", "tris5", "tris17", "tris4000", "stacked", "blob_spheres",
                                  "pathlines"])
def test_the_wide_walk_gives_the_binary_walks_hits(hip, kind):
    from galaxy_amd import lib as glib
    L = glib.lib()
    B = scenes.build_scene(hip, _scene(kind))
    hr = _rays()
    for k, typ in ((1, abi.RAY_SHADOW), (2, abi.RAY_AO)):
        hr["type"][k::5] = typ
    geom, prim = glib.DeviceArray(4 * hr.n), glib.DeviceArray(4 * hr.n)
    glib.check(L.gxy_model_set_hit_output(B.vis.model, geom.ptr, prim.ptr))
    got = []
    try:
        for width, stack, waves in ((2, 16, 0), (2, 0, 8), (4, 0, 0), (2, 0, 0)):
            glib.check(L.gxy_set_bvh_width(width))
            glib.check(L.gxy_set_geometry_stack(stack))
            glib.check(L.gxy_set_geometry_waves(waves))
            d = glib.DeviceRays.from_host(hr)
            assert hip.trace(B.vis, d) == ""
            g = d.download()
            got.append([g[f].view(np.int32) for f in abi.FIELDS] + [geom.to_host(np.int32, hr.n),
                                                                   prim.to_host(np.int32, hr.n)])
    finally:
        L.gxy_set_bvh_width(2)
        L.gxy_set_geometry_stack(0)
        L.gxy_set_geometry_waves(0)
        L.gxy_model_set_hit_output(B.vis.model, None, None)
    assert (got[0][-2] >= 0).any()
    for other in got[1:]:
        for f, a, b in zip(abi.FIELDS + ("geom", "prim"), got[0], other):
            bad = np.nonzero(a != b)[0]
            assert len(bad) == 0, (kind, f, bad[:5])


def test_mixed_scenes_take_the_same_walks(hip):
    """A volume with a mesh inside (the kernel that both marches and walks)."""
    from galaxy_amd import lib as glib
    L = glib.lib()
    sc = workloads.unit_volume_scene(24, 4)
    sc.meshes = [scenes.blob_mesh(4000, 9)]
    B = scenes.build_scene(hip, sc)
    hr = _rays()
    got = []
    try:
        for width, stack in ((2, 16), (4, 0)):
            glib.check(L.gxy_set_bvh_width(width))
            glib.check(L.gxy_set_geometry_stack(stack))
            d = glib.DeviceRays.from_host(hr.subset(np.arange(900)))
            assert hip.trace(B.vis, d) == ""
            g = d.download()
            got.append([g[f].view(np.int32) for f in abi.FIELDS])
    finally:
        L.gxy_set_bvh_width(2)
        L.gxy_set_geometry_stack(0)
    assert all(np.array_equal(a, b) for a, b in zip(*got))


def _closest(hip, B, hr, width, stack):
    from galaxy_amd import lib as glib
    L = glib.lib()
    geom, prim = glib.DeviceArray(4 * hr.n), glib.DeviceArray(4 * hr.n)
    glib.check(L.gxy_model_set_hit_output(B.vis.model, geom.ptr, prim.ptr))
    try:
        glib.check(L.gxy_set_bvh_width(width))
        glib.check(L.gxy_set_geometry_stack(stack))
        d = glib.DeviceRays.from_host(hr)
        assert hip.trace(B.vis, d) == ""
        return d.download()["t"], geom.to_host(np.int32, hr.n), prim.to_host(np.int32, hr.n)
    finally:
        L.gxy_set_bvh_width(2)
        L.gxy_set_geometry_stack(0)
        L.gxy_model_set_hit_output(B.vis.model, None, None)


@pytest.mark.parametrize("sign", [1, -1])
def test_directions_whose_reciprocal_nearly_overflows(hip, sign):
    """1/d is finite, its product with the walk's far-plane factor is not."""
    B = scenes.build_scene(hip, _scene("blob_spheres"))
    rng = np.random.default_rng(4)
    n = 2000
    o, d = rng.uniform(-0.2, 1.2, (n, 3)), rng.normal(size=(n, 3))
    least = 1.0 / np.float64(np.finfo(f32).max)          # the smallest d with a finite 1/d
    for a in range(3):
        d[a::3, a] = sign * least * rng.uniform(1.0000002, 1.000001, len(d[a::3]))
    hr = abi.HostRays.from_arrays(o.astype(f32), d.astype(f32), np.zeros(n, f32), np.full(n, 1e30, f32))
    want, got = _closest(hip, B, hr, 2, 16), _closest(hip, B, hr, 4, 0)
    assert (want[1] >= 0).sum() > 200
    for a, b in zip(want, got):
        assert np.array_equal(a.view(np.int32), b.view(np.int32)), np.nonzero(a != b)[0][:5]


@pytest.mark.parametrize("spheres", [3, 11, 18, 27, 40])
def test_rays_that_skip_every_axis_find_all_children(hip, spheres):
    """Origin over direction overflows on all axes: every slot of a node is
    entered, the empty ones of nodes with fewer than four children too."""
    rng = np.random.default_rng(spheres)
    at, unit = 1e20, 1.4e14                              # (floats near 1e20 are 8.8e12 apart)
    c = at + unit * rng.integers(0, 5, (spheres, 3))
    box = ((at - 10 * unit,) * 3, (at + 15 * unit,) * 3)
    sc = scenes.SceneDesc(local_box=box, global_box=box, spheres=[scenes.SpheresDesc(
        c.astype(f32), rng.uniform(0, 1, spheres).astype(f32), 0.5 * unit, 0.7 * unit, 0.0, 1.0)])
    B = scenes.build_scene(hip, sc)
    n = 1000
    o = at + unit * rng.integers(-8, 14, (n, 3))
    d = c[rng.integers(spheres, size=n)] - o + 0.2 * unit * rng.normal(size=(n, 3))
    d *= 1e-19 / np.linalg.norm(d, axis=1, keepdims=True)
    hr = abi.HostRays.from_arrays(o.astype(f32), d.astype(f32), np.zeros(n, f32), np.full(n, np.inf, f32))
    want, got = _closest(hip, B, hr, 2, 16), _closest(hip, B, hr, 4, 0)
    assert (want[1] >= 0).sum() > 100
    for a, b in zip(want, got):
        assert np.array_equal(a.view(np.int32), b.view(np.int32)), np.nonzero(a != b)[0][:5]


def _line_scene(levels, seed):
    """Overlapping triangles that halve in size along a line: a tree of about
    `levels` levels, most of whose boxes a ray along the line enters."""
    rng = np.random.default_rng([levels, seed])
    x = 0.5 ** np.arange(levels)
    c = np.c_[x, 0 * x, 0 * x] + 0.2 * x[:, None] * rng.uniform(-1, 1, (levels, 3))
    v = c[:, None] + 1.5 * x[:, None, None] * rng.uniform(-0.5, 0.5, (levels, 3, 3))
    box = ((-4.0,) * 3, (4.0,) * 3)
    return scenes.SceneDesc(local_box=box, global_box=box, meshes=[scenes.MeshDesc(
        v.reshape(-1, 3).astype(f32), np.arange(3 * levels, dtype=np.uint32).reshape(-1, 3))])


def test_every_stack_holds_its_trees(hip):
    """Trees around the depths at which an LDS stack setting still holds them, and
    up to 60 levels: private entries, the 4-wide walk at its bound of 26 levels, and
    the binary walk beyond it."""
    from batch_scenes import graded_scene, rays_at_triangles
    L = hip.L
    depths = set()
    scs = [_line_scene(k, s) for k in range(12, 37) for s in range(3)] + [graded_scene(s) for s in range(6)]
    for sc in scs:
        B = scenes.build_scene(hip, sc)
        a, b, depth, sah = C.c_int(), C.c_int(), C.c_int(), C.c_float()
        assert L.gxy_model_bvh_stats(B.vis.model, C.byref(a), C.byref(b), C.byref(depth), C.byref(sah)) == 0
        depths.add(depth.value)
        hr = rays_at_triangles(sc, 3000, 2)
        rng = np.random.default_rng(1)
        for f in ("oy", "oz"):                           # along the line of the triangles, both ways
            hr[f][:600] = rng.uniform(-0.02, 0.02, 600)
        hr["ox"][:600] = np.where(np.arange(600) % 2, 2.0, -1.0)
        hr["dx"][:600] = np.where(np.arange(600) % 2, -1.0, 1.0)
        for f in ("dy", "dz"):
            hr[f][:600] = rng.uniform(-0.01, 0.01, 600)
        hr["type"][::3] = abi.RAY_SHADOW
        want = _closest(hip, B, hr, 2, 0)
        assert (want[1] >= 0).sum() > 1000
        for width, stack in ((2, 16), (2, 24), (2, 32), (4, 0)):
            got = _closest(hip, B, hr, width, stack)
            for x, y in zip(want, got):
                assert np.array_equal(x.view(np.int32), y.view(np.int32)), (depth.value, width, stack)
    for stack in (16, 24, 32):
        assert {stack - 2, stack - 1} <= depths, sorted(depths)
    assert max(depths) >= 55
