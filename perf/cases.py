"""The calls whose speed matters to a user of this library, as measurable cases.

A case is one call (or the fixed sequence of calls) that a program makes per
frame, per ray list or per time step once its scene is resident on the GPU:

  frame    gxy_render_frame over a volume, a triangle mesh, icospheres, data
           spheres or path lines
  sample   gxy_sample_raylist: particles at the isovalue crossings of random rays
  pass     one RayList through the separate entry points that a renderer's own
           pass loop binds (TraceRays_*, gxy_spawn_offsets, gxy_classify, ...)
  batch    gxy_batch_run: many uneven ray lists over many resident datasets
  step     a new time step of a deforming mesh: build its model, render it
  serve    gxy_server_run: a burst of render and sample requests at once

The sizes are those of bench.py and galaxy_amd/workloads.py (512^3 volume at
1920x1080, 20 K-triangle sphere at 512x512, nine icospheres at 3840x2160 with
16 AO rays, 4000 path lines at 1024x1024, 1 K - 1 M-ray lists) and the small
and ragged ones that viewers and tests use.  Process-wide settings stay at the
library's defaults, apart from those a workload states (the early-termination
alpha, the AO directions), which are set before each call as a program that
holds several scenes would.
"""
import ctypes as C
import functools
import math

import numpy as np
import torch

from galaxy_amd import abi, lib as glib, scenes, serve, workloads

f32 = np.float32
NO_NEIGHBORS = np.full(6, -1, np.int32)
TWO_COLORS = np.array([[0.0, 0.9, 0.4, 0.3], [1.0, 0.3, 0.6, 0.9]], f32)


# --------------------------------------------------------------------- the cases
def frame(name, scene, width, height, **kw):
    c = dict(call="frame", scene=scene, width=width, height=height, lights=1, shadows=True, n_ao=0, alpha=0.999)
    if name:
        c["name"] = name
    return c | kw


def volume(nx, ny, nz, layout, isovalues=1, slices=0, dvr=True, octaves=4):
    return dict(nx=nx, ny=ny, nz=nz, layout=layout, isovalues=isovalues, slices=slices, dvr=dvr, octaves=octaves)


def listed():
    return [
        # a viewer's thumbnail of a small field while the camera moves: launches and host waits count
        frame("volume_preview_128", "volume", 128, 128, **volume(64, 64, 64, 0)),
        # a viewer window over a ragged field with a slice, two isosurfaces, two lights and AO
        frame("volume_viewer_800x600", "volume", 800, 600, lights=2, n_ao=8, **volume(201, 157, 120, 0, 2, 1)),
        # the headline volume render: full HD, 512^3 in the bricked layout its benchmark settles on
        frame("volume_1080p_512", "volume", 1920, 1080, alpha=0.99, **volume(512, 512, 512, 4)),
        # one small closed mesh, 20 K triangles, with a hard shadow
        frame("mesh_512", "mesh", 512, 512, triangles=20480),
        # the largest geometry frame: 11.8 M triangles, 4K, 16 ambient-occlusion rays per hit
        frame("icospheres_4k_ao16", "icospheres", 3840, 2160, n_ao=16, subdiv=8),
        # particles of a simulation step as data-driven spheres, with AO
        frame("spheres_1024_ao4", "spheres", 1024, 1024, n_ao=4, spheres=200_000),
        # stream lines of a flow field as data-driven tubes
        frame("pathlines_1024", "pathlines", 1024, 1024, lines=4000, verts=64),
        # isovalue particles for an in-situ sampler: a million random rays
        dict(name="sample_1m_256", call="sample", rays=1_000_000, edge=256, layout=4),
        # one list of a renderer that drives the pass itself, over a volume with a mesh inside
        dict(name="pass_100k", call="pass", rays=100_003, edge=96, triangles=50_000, n_ao=2),
        # many uneven lists over many datasets, shadow and 2 AO rays per hit, in one call
        dict(name="batch_64_lists", call="batch", lists=64, datasets=16, max_rays=1_000_000, max_edge=384,
             max_triangles=1_000_000),
        # in-situ geometry: a mesh that deforms every time step is rebuilt and shown
        dict(name="step_mesh_1m", call="step", triangles=1_000_000, width=512, height=512),
        # a burst of requests at a render server
        dict(name="serve_12_requests", call="serve", requests=12, edge=256, triangles=1_000_000, max_pixels=1920 * 1080,
             max_rays=2_000_000),
    ]


def draw(rng):
    def logu(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def size(lo, hi):
        px, aspect = logu(lo * lo, hi * hi), rng.choice([1.0, 4 / 3, 16 / 9])
        h = max(8, int(round(math.sqrt(px / aspect))))
        return max(8, int(round(h * aspect)) + rng.randrange(2)), h

    kind = rng.choice(["volume", "volume", "volume", "mesh", "icospheres", "spheres", "pathlines", "sample", "pass",
                       "batch", "step", "serve"])
    if kind == "volume":
        w, h = size(96, 1440)
        e = logu(32, 448)
        dims = [max(16, int(round(e * rng.uniform(0.6, 1.1)))) for _ in range(3)]
        return frame(None, "volume", w, h, lights=rng.randint(1, 2), shadows=rng.random() < 0.8,
                     n_ao=rng.choice([0, 0, 4]), alpha=rng.choice([0.99, 0.999]),
                     **volume(*dims, rng.choice([0, 4, 8]), rng.randint(0, 2), rng.choice([0, 0, 1]),
                              octaves=rng.randint(2, 4)))
    if kind == "mesh":
        w, h = size(128, 2048)
        return frame(None, "mesh", w, h, lights=rng.randint(1, 2), n_ao=rng.choice([0, 0, 8]),
                     triangles=logu(2_000, 2_000_000))
    if kind == "icospheres":
        w, h = size(256, 2048)
        return frame(None, "icospheres", w, h, n_ao=rng.choice([1, 4, 16]), subdiv=rng.randint(3, 7))
    if kind == "spheres":
        w, h = size(128, 1440)
        return frame(None, "spheres", w, h, n_ao=rng.choice([0, 4]), spheres=logu(1_000, 1_000_000))
    if kind == "pathlines":
        w, h = size(128, 1440)
        return frame(None, "pathlines", w, h, lines=logu(50, 5_000), verts=rng.randint(8, 80))
    if kind == "sample":
        return dict(call="sample", rays=logu(1_000, 2_000_000), edge=logu(48, 400), layout=rng.choice([0, 4, 8]))
    if kind == "pass":
        return dict(call="pass", rays=logu(500, 1_000_000), edge=logu(32, 256), triangles=logu(2_000, 500_000),
                    n_ao=rng.choice([0, 2, 8]))
    if kind == "batch":
        return dict(call="batch", lists=rng.randint(8, 64), datasets=rng.randint(2, 12), max_rays=logu(10_000, 1_000_000),
                    max_edge=rng.randint(130, 320), max_triangles=logu(60_000, 1_000_000))
    if kind == "step":
        w, h = size(128, 1024)
        return dict(call="step", triangles=logu(5_000, 900_000), width=w, height=h)
    return dict(call="serve", requests=rng.randint(2, 12), edge=logu(96, 320), triangles=logu(50_000, 1_000_000),
                max_pixels=logu(300 * 300, 1920 * 1080), max_rays=logu(1_200_000, 2_000_000))


# --------------------------------------------------------------------- scenes
@functools.lru_cache(maxsize=8)
def base_icosphere(subdiv):
    return scenes.icosphere(subdiv, 0.45)


@functools.lru_cache(maxsize=8)
def base_sphere_grid(triangles):
    """Unit directions and triangles of a UV sphere of about `triangles` triangles."""
    nlat = max(4, int(round((triangles / 4.0) ** 0.5)))
    nlon = 2 * nlat
    th = np.linspace(0, np.pi, nlat + 1)[:, None]
    ph = np.linspace(0, 2 * np.pi, nlon, endpoint=False)[None, :]
    n = np.stack(np.broadcast_arrays(np.sin(th) * np.cos(ph), np.sin(th) * np.sin(ph), np.cos(th)), -1)
    return n.reshape(-1, 3), scenes.uv_grid_indices(nlon, nlat)


def bumpy_sphere(triangles, rng, radius=1.0, amp=0.06, center=(0.0, 0.0, 0.0)):
    """A sphere whose radius swings with three seeded waves of the direction."""
    n, idx = base_sphere_grid(triangles)
    f = np.zeros(len(n))
    for k in range(3):
        f += np.sin((k + 2) * (n @ rng.normal(size=3)) + rng.uniform(0, 6.28)) / (k + 1)
    v = (n * (radius * (1.0 + amp * f))[:, None] + np.asarray(center)).astype(f32)
    data = ((f - f.min()) / max(1e-9, f.max() - f.min())).astype(f32)
    return scenes.MeshDesc(v, idx, n.astype(f32), data, TWO_COLORS)


def lighting(case, rng):
    src = [[3.0 + rng.uniform(-0.5, 0.5), 4.0, 5.0], [-4.0, 2.0 + rng.uniform(-0.5, 0.5), 3.0]][:case.get("lights", 1)]
    return scenes.LightingDesc(np.array(src, f32), np.full(len(src), 2, np.int32), Ka=0.3, Kd=0.7,
                               n_ao=case.get("n_ao", 0), ao_radius=0.5, shadows=case.get("shadows", True))


def orbit(rng, dist, lift, aov, width, height, center=(0.0, 0.0, 0.0)):
    az, el = rng.uniform(0, 2 * math.pi), lift + rng.uniform(-0.15, 0.15)
    eye = (center[0] + dist * math.cos(el) * math.sin(az), center[1] + dist * math.sin(el),
           center[2] + dist * math.cos(el) * math.cos(az))
    return scenes.CameraDesc(eye, center, (0.0, 1.0, 0.0), aov, width, height)


def volume_scene(case, seed, rng):
    dims = (case["nx"], case["ny"], case["nz"])
    d = f32(2.0 / (max(dims) - 1))
    origin = tuple(f32(-0.5 * float(d) * (n - 1)) for n in dims)
    lbox, gbox = workloads.volume_boxes(dims, origin, (d,) * 3)
    vol = scenes.VolumeDesc(None, origin, (d,) * 3, sampling_rate=0.5, local_box=lbox, global_box=gbox, shape=dims,
                            noise=(seed & 0x7FFFFFFF, case["octaves"], 4.0))
    x = np.linspace(0.0, 1.0, 8)
    rgb, op = workloads.VOLUME_RENDER_TF
    vv = scenes.VolumeVisDesc(vol, colormap=np.c_[x, rgb].astype(f32), opacitymap=np.c_[x, op].astype(f32),
                              isovalues=np.array([0.5, 0.62][:case["isovalues"]], f32), volume_render=case["dvr"])
    if case["slices"]:
        vv.slices = np.array([[0.0, 0.0, 1.0, rng.uniform(-0.2, 0.2)]], f32)
    return scenes.SceneDesc(volume_vis=[vv], local_box=lbox, global_box=gbox)


def frame_scene(case, seed):
    """(SceneDesc with its lighting and one camera) of a frame case."""
    rng = np.random.default_rng(seed)
    w, h, kind = case["width"], case["height"], case["scene"]
    if kind == "volume":
        sc = volume_scene(case, seed, rng)
        cam = orbit(rng, 3.9, 0.42, 35.0, w, h)
    elif kind == "mesh":
        sc = scenes.SceneDesc(meshes=[bumpy_sphere(case["triangles"], rng)], local_box=((-1.5,) * 3, (1.5,) * 3),
                              global_box=((-1.5,) * 3, (1.5,) * 3))
        cam = orbit(rng, 3.2, 0.1, 45.0, w, h)
    elif kind == "icospheres":
        base, meshes = base_icosphere(case["subdiv"]), []
        for k in range(9):
            c = np.array([(k // 3 - 1) * 1.1, (k % 3 - 1) * 1.1, rng.uniform(-0.05, 0.05)], f32)
            meshes.append(scenes.MeshDesc(base.vertices + c, base.indices, base.normals, base.vertex_data, TWO_COLORS))
        box = ((-1.8, -1.8, -0.6), (1.8, 1.8, 0.6))
        sc = scenes.SceneDesc(meshes=meshes, local_box=box, global_box=box)
        cam = scenes.CameraDesc((rng.uniform(-0.2, 0.2), -1.2, 4.2), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 50.0, w, h)
    elif kind == "spheres":
        n = case["spheres"]
        p = rng.uniform(0.0, 1.0, (n, 3))
        p += 0.05 * np.sin(2 * math.pi * p[:, [1, 2, 0]])
        r = 0.35 * n ** (-1.0 / 3.0)
        sc = scenes.SceneDesc(spheres=[scenes.SpheresDesc(p.astype(f32), rng.uniform(0, 1, n).astype(f32), 0.5 * r, r,
                                                          0.0, 1.0, TWO_COLORS)],
                              local_box=((-0.2,) * 3, (1.2,) * 3), global_box=((-0.2,) * 3, (1.2,) * 3))
        cam = orbit(rng, 2.2, 0.3, 40.0, w, h, (0.5, 0.5, 0.5))
    else:
        sc, _ = workloads.pathlines(w, h, case["lines"], case["verts"], seed)
        cam = orbit(rng, 1.9, 0.1, 35.0, w, h, (0.5, 0.5, 0.5))
    sc.lighting = lighting(case, rng)
    sc.cameras = [cam]
    return sc


class Scene:
    """A scene resident on the GPU; its objects are given back with it."""

    def __init__(self, desc, layout=0):
        self.desc = desc
        self.hip = glib.HipBackend()
        self.built = scenes.build_scene(self.hip, desc, scenes.resolve_lights(desc.lighting, desc.cameras[0])
                                        if desc.cameras else None)
        if layout:
            glib.check(self.hip.L.gxy_volume_set_layout(self.built.handles[0], layout), "volume_set_layout")

    def __del__(self):
        L = glib.load()
        for h in self.built.handles:
            for fn in (L.gxy_model_destroy, L.gxy_volume_destroy, L.gxy_tf_destroy):
                fn(h)
        self.built.handles = []


class Rays:
    """A RayList whose 25 arrays are rows of two torch tensors."""

    def __init__(self, n):
        self.n = n
        m = max(16, (n + 15) // 16 * 16)
        self.f = torch.zeros(len(abi.FLOAT_FIELDS), m, dtype=torch.float32, device="cuda")
        self.i = torch.zeros(len(abi.INT_FIELDS), m, dtype=torch.int32, device="cuda")
        rows = dict(zip(abi.FLOAT_FIELDS, self.f)) | dict(zip(abi.INT_FIELDS, self.i))
        self.ispc = abi.RayList_ispc(**{k: v.data_ptr() for k, v in rows.items()})
        self.rows = rows


def stats_array(st):
    return np.array([st.primary_rays, st.secondary_rays, st.ray_passes, st.terminated, st.dropped, st.kept, st.samples],
                    np.int64)


# --------------------------------------------------------------------- prepare
def prepare(case, seed):
    glib.lib()
    torch.zeros(1, device="cuda")
    return globals()["prepare_" + case["call"]](case, seed)


def camera_args(cam):
    return [glib.a3(cam.eye), glib.a3(cam.center), glib.a3(cam.up)]


def prepare_frame(case, seed):
    s = Scene(frame_scene(case, seed), case.get("layout", 0))
    cam = s.desc.cameras[0]
    return dict(case=case, scene=s, cam=cam, cam3=camera_args(cam), stats=abi.FrameStats(),
                ao=(1, workloads.NINE_ICOSPHERES_AO_SEED) if case["scene"] == "icospheres" else (0, 0),
                fb=torch.zeros(cam.height, cam.width, 4, dtype=torch.float32, device="cuda"))


def prepare_sample(case, seed):
    s = Scene(workloads.unit_volume_scene(case["edge"], seed & 0x7FFFFFFF), case["layout"])
    n = case["rays"]
    cap = 8 * n + 1024
    return dict(case=case, scene=s, rays=Rays(n), seed=seed & 0x7FFFFFFF, capacity=cap, stats=abi.FrameStats(),
                lo=glib.a3((0, 0, 0)), hi=glib.a3((1, 1, 1)),
                xyz=torch.zeros(cap, 3, dtype=torch.float32, device="cuda"))


def prepare_pass(case, seed):
    rng = np.random.default_rng(seed)
    sc = workloads.unit_volume_scene(case["edge"], seed & 0x7FFFFFFF)
    sc.meshes = [bumpy_sphere(case["triangles"], rng, 0.3, 0.06, (0.5, 0.5, 0.5))]
    sc.lighting = lighting(dict(case, shadows=True), rng)
    s = Scene(sc)
    n = case["rays"]
    side = int(math.ceil(math.sqrt(n)))
    return dict(case=case, scene=s, rays=Rays(n), children=Rays(n * (case["n_ao"] + 1)), keep=Rays(n), side=side,
                seed=seed & 0x7FFFFFFF, lo=glib.a3((0, 0, 0)), hi=glib.a3((1, 1, 1)),
                offsets=torch.zeros(2, max(1, n), dtype=torch.int32, device="cuda"),
                fb=torch.zeros(side, side, 4, dtype=torch.float32, device="cuda"))


class BatchScene:
    def __init__(self, case, seed):
        L = glib.lib()
        descs, lists, light = workloads.batched_lists(case["lists"], case["datasets"], (1_000, case["max_rays"]),
                                                      (128, case["max_edge"]), (50_000, case["max_triangles"]))
        self.scenes = [Scene(workloads.dataset_scene((kind, size, sd + seed % 999983)), 4 if kind == "volume" else 0)
                       for kind, size, sd in descs]
        self.keep = []
        self.h = glib.checkp(L.gxy_batch_create(256), "batch_create")
        ids = [glib.check(L.gxy_batch_add_dataset(self.h, C.byref(s.built.vis), 0.001)) for s in self.scenes]
        lights = scenes.make_lighting(light, self.keep)
        glib.check(L.gxy_batch_set_lighting(self.h, C.byref(lights), 0.001), "batch_set_lighting")
        self.keep.append(lights)
        self.fb = torch.zeros(sum(n for n, _, _ in lists), 4, dtype=torch.float32, device="cuda")
        lo, hi, at = glib.a3((0, 0, 0)), glib.a3((1, 1, 1)), 0
        for n, ds, sd in lists:
            d = glib.DeviceRays(n)
            k = glib.check(L.gxy_batch_add_list(self.h, ids[ds], abi.BATCH_RENDER, n, C.byref(d.ispc),
                                                self.fb[at:].data_ptr(), n, 1, None, 0, None), "batch_add_list")
            glib.check(L.gxy_batch_set_list_seed(self.h, k, sd + seed % 1000, lo.ctypes.data, hi.ctypes.data))
            self.keep.append(d)
            at += n

    def __del__(self):
        if self.h:
            glib.load().gxy_batch_destroy(self.h)
            self.h = None


def prepare_batch(case, seed):
    return dict(case=case, batch=BatchScene(case, seed), stats=abi.BatchStats())


def prepare_step(case, seed):
    rng = np.random.default_rng(seed)
    mesh = bumpy_sphere(case["triangles"], rng)
    cam = orbit(rng, 3.2, 0.1, 45.0, case["width"], case["height"])
    box = ((-1.5,) * 3, (1.5,) * 3)
    sc = scenes.SceneDesc(local_box=box, global_box=box, lighting=lighting(dict(shadows=True), rng), cameras=[cam])
    s = Scene(sc)
    s.tf = s.hip.tf_create_from_maps(TWO_COLORS, scenes.DEFAULT_OPACITYMAP.copy(), None)
    s.built.handles.append(s.tf)
    return dict(case=case, scene=s, mesh=mesh, cam=cam, cam3=camera_args(cam), stats=abi.FrameStats(),
                fb=torch.zeros(cam.height, cam.width, 4, dtype=torch.float32, device="cuda"))


class ServeScene:
    def __init__(self, case, seed):
        rng = np.random.default_rng(seed)
        e = case["edge"]
        descs = [workloads.unit_volume_scene(e, seed & 0x7FFFFFFF), workloads.unit_volume_scene(e * 3 // 4, 1 + seed % 999983),
                 scenes.SceneDesc(meshes=[bumpy_sphere(case["triangles"], rng, 0.35, 0.06, (0.5,) * 3)],
                                  local_box=workloads.UNIT_BOX, global_box=workloads.UNIT_BOX)]
        self.scenes = [Scene(d, 4 if d.volume_vis else 0) for d in descs]
        self.server = serve.Server(32 << 30, 64, 256)
        for s in self.scenes:
            self.server.add_dataset(s.built)
        self.keep = []
        self.server.set_lighting(scenes.make_lighting(workloads.batch_lighting(), self.keep))
        self.server.set_step_rays(4_000_000)
        # one mix of kinds and sizes per case; views and ray seeds from the seed
        self.reqs, outs = serve.request_stream(case["requests"], 200.0, 0.5, np.random.default_rng(5),
                                               (128 * 128, case["max_pixels"]), (20_000, case["max_rays"]), (0, 1),
                                               (0, 1, 2), keep_outputs=True)
        for r in self.reqs:
            r.arrival = 0.0
            r.eye[:] = list(serve.orbit_eye(rng))
            r.seed = int(rng.integers(1 << 30))
            if r.kind == 1:      # particles arrive in no fixed order: only their count is taken
                r.out = None
        self.images = [o for r, o in zip(self.reqs, outs) if r.kind == 0]

    def __del__(self):
        self.server.destroy()


def prepare_serve(case, seed):
    return dict(case=case, serve=ServeScene(case, seed))


# --------------------------------------------------------------------- run
def run(state):
    return globals()["run_" + state["case"]["call"]](state)


def render(L, state):
    s, cam, case = state["scene"], state["cam"], state["case"]
    glib.check(L.gxy_set_opacity_threshold(case.get("alpha", 0.999)))
    glib.check(L.gxy_set_ao_directions(*state.get("ao", (0, 0))))
    fb, st = state["fb"], state["stats"]
    eye, cen, up = state["cam3"]
    glib.check(L.gxy_memset(fb.data_ptr(), 0, fb.numel() * 4), "memset")
    glib.check(L.gxy_render_frame(C.byref(s.built.vis), C.byref(s.built.lights), eye.ctypes.data, cen.ctypes.data,
                                  up.ctypes.data, cam.aov, cam.width, cam.height, NO_NEIGHBORS.ctypes.data, 0.001,
                                  1 << 30, fb.data_ptr(), C.byref(st)), "render_frame")
    return {"image": fb, "counts": stats_array(st)}


def run_frame(state):
    return render(glib.lib(), state)


def run_sample(state):
    L, r, st = glib.lib(), state["rays"], state["stats"]
    count = C.c_int(0)
    glib.check(L.gxy_rays_random(C.byref(r.ispc), r.n, state["seed"], r.n, abi.RAY_PRIMARY, state["lo"].ctypes.data,
                                 state["hi"].ctypes.data), "rays_random")
    glib.check(L.gxy_sample_raylist(C.byref(state["scene"].built.vis), r.n, C.byref(r.ispc), 1 << 30,
                                    state["xyz"].data_ptr(), state["capacity"], C.byref(count), C.byref(st)),
               "sample_raylist")
    return {"particles": state["xyz"], "count": count.value, "counts": stats_array(st)}


def run_pass(state):
    """TraceRays::Trace and the work around it, call by call."""
    L, case, s = glib.lib(), state["case"], state["scene"]
    r, out, keep, n = state["rays"], state["children"], state["keep"], state["rays"].n
    rays, lights, nao = C.byref(r.ispc), C.byref(s.built.lights), case["n_ao"]
    ao, sh = state["offsets"][0].data_ptr(), state["offsets"][1].data_ptr()
    fb, side = state["fb"], state["side"]
    glib.check(L.gxy_set_opacity_threshold(0.999))
    glib.check(L.gxy_set_ao_directions(0, 0))
    glib.check(L.gxy_rays_random(rays, n, state["seed"], side, abi.RAY_PRIMARY, state["lo"].ctypes.data,
                                 state["hi"].ctypes.data), "rays_random")
    glib.check(L.gxy_memset(fb.data_ptr(), 0, fb.numel() * 4), "memset")
    L.TraceRays_TraceRays(None, C.byref(s.built.vis), n, rays, 0.001)
    n_ao, n_sh = C.c_int(0), C.c_int(0)
    glib.check(L.gxy_spawn_offsets(n, rays, nao, 1, 1, ao, sh, C.byref(n_ao), C.byref(n_sh)), "spawn_offsets")
    L.TraceRays_ambientLighting(None, lights, n, rays)
    if n_ao.value:
        L.TraceRays_generateAORays(None, lights, n, rays, ao, C.byref(out.ispc), 0.001)
    L.TraceRays_diffuseLighting(None, lights, n, rays)
    if n_sh.value:
        L.TraceRays_generateShadowRays(None, lights, n, rays, sh, C.byref(out.ispc), 0.001)
    glib.check(L.gxy_classify(n, rays, 1), "classify")
    glib.check(L.gxy_assign_destinations(n, rays, C.byref(s.built.vis.local_bb), NO_NEIGHBORS.ctypes.data, 1))
    glib.check(L.gxy_accumulate_terminated(n, rays, fb.data_ptr(), side, side), "accumulate")
    counts = (C.c_int * 1)()
    glib.check(L.gxy_partition_rays(n, rays, 0, None, C.byref(keep.ispc), counts), "partition")
    kids = [out.rows[k] for k in ("ox", "oy", "oz", "dx", "dy", "dz", "r", "g", "b", "tMax")]
    return {"image": fb, "rays": [r.rows[k] for k in ("t", "r", "g", "b", "o")], "children": kids,
            "pixels": [out.rows[k] for k in ("x", "y", "type")], "spawned": [n_ao.value, n_sh.value, counts[0]],
            "states": [r.rows[k] for k in ("term", "classification")]}


def run_batch(state):
    L, b, st = glib.lib(), state["batch"], state["stats"]
    glib.check(L.gxy_set_opacity_threshold(0.999))
    glib.check(L.gxy_set_ao_directions(0, 0))
    glib.check(L.gxy_batch_run(b.h, 2, C.byref(st)), "batch_run")
    return {"images": b.fb, "counts": np.array([st.rays, st.samples, st.spawned, st.terminated, st.dropped, st.kept],
                                               np.int64)}


def run_step(state):
    s, m = state["scene"], state["mesh"]
    L = s.hip.L
    model = s.hip.model_create()
    s.hip.model_add_triangles(model, m.vertices, m.indices, m.normals, m.vertex_data, s.tf)
    s.hip.model_commit(model)
    s.built.vis.model = model
    out = render(L, state)
    s.built.vis.model = None
    glib.check(L.gxy_model_destroy(model), "model_destroy")
    return out


def run_serve(state):
    L, sv = glib.lib(), state["serve"]
    glib.check(L.gxy_set_opacity_threshold(0.999))
    glib.check(L.gxy_set_ao_directions(0, 0))
    res, st = sv.server.run(sv.reqs, abi.SERVE_CONTINUOUS)
    return {"images": sv.images, "particles": np.array([r.particles for r in res], np.int64),
            "rays": np.array([r.rays for r in res], np.int64), "status": np.array([r.status for r in res], np.int64),
            "totals": np.array([st.rays, st.samples], np.int64)}


# --------------------------------------------------------------------- work
RAY = 104           # bytes of a traced ray's fields read and written
SAMPLE = 36         # flops of a trilinear volume sample with its position
WALK = 1000         # flops of a ray's walk through a tree over a mesh of this size and its primitive tests


def work(case):
    """Bytes: the scene once, each primary ray's fields and the image once.
    Flops: samples along the rays (half the box's depth at two samples per
    voxel for primary rays) or tree walks, with half the pixels on the scene."""
    call = case["call"]
    if call in ("frame", "step"):
        px = case["width"] * case["height"]
        hits = 0.3 * px
        rays = 0.5 * px + hits * (case.get("n_ao", 0) + case.get("lights", 1))
        if case.get("scene") == "volume":
            depth = max(case["nx"], case["ny"], case["nz"])
            return {"bytes": 4.0 * case["nx"] * case["ny"] * case["nz"] + 16.0 * px + RAY * rays,
                    "flops": SAMPLE * 0.5 * depth * rays}
        scene = {"mesh": 24 * case.get("triangles", 0), "icospheres": 9 * 24 * 20 * 4 ** case.get("subdiv", 0),
                 "spheres": 16 * case.get("spheres", 0), "pathlines": 16 * case.get("lines", 0) * case.get("verts", 0),
                 None: 48 * case.get("triangles", 0)}[case.get("scene")]
        return {"bytes": float(scene) + 16.0 * px + RAY * rays, "flops": WALK * rays}
    if call == "sample":
        return {"bytes": 4.0 * case["edge"] ** 3 + RAY * case["rays"] + 24.0 * case["rays"],
                "flops": SAMPLE * 1.2 * case["edge"] * case["rays"]}
    if call == "pass":
        n = case["rays"]
        return {"bytes": 4.0 * case["edge"] ** 3 + 24.0 * case["triangles"] + (RAY + 64 * (0.5 * case["n_ao"] + 0.5)) * n,
                "flops": SAMPLE * 0.3 * case["edge"] * n + WALK * n}
    if call == "batch":
        _, lists, _ = workloads.batched_lists(case["lists"], case["datasets"], (1_000, case["max_rays"]))
        n = sum(x[0] for x in lists)
        return {"bytes": RAY * 2.0 * n + case["datasets"] * 4.0 * 220 ** 3, "flops": 2.0 * n * SAMPLE * 60}
    n = case["requests"] * (0.25 * case["max_pixels"] + 0.25 * case["max_rays"])
    return {"bytes": RAY * n + 4.0 * 1.5 * case["edge"] ** 3, "flops": n * SAMPLE * 0.5 * case["edge"]}


# --------------------------------------------------------------------- the same volume frame in 64 bits
def exact(case, seed):
    """The image of a volume frame in float64: camera, march, isosurfaces,
    lighting and shadow rays restated in torch.  Slices and AO are left to the
    bounds on the float32 outputs, as are the calls whose outputs are closest
    hits over large scenes."""
    if case["call"] != "frame" or case["scene"] != "volume" or case["slices"] or case["n_ao"]:
        return None
    sc = frame_scene(case, seed)
    vol = sc.volume_vis[0].volume
    s = Scene(sc)
    vox = torch.from_numpy(s.hip.volume_download(s.built.handles[0], vol.dims)).cuda().double()
    return {"image": ExactVolumeFrame(sc, vox, case["alpha"]).image(), "counts": None}


def vec(a):
    return torch.tensor([float(x) for x in a], dtype=torch.float64, device="cuda")


def unit(v):
    return v / v.norm(dim=-1, keepdim=True)


class ExactVolumeFrame:
    def __init__(self, sc, vox, alpha, eps=0.001):
        vv = sc.volume_vis[0]
        self.sc, self.vox, self.alpha, self.eps = sc, vox, alpha, eps
        self.lo, self.hi = vec(sc.local_box[0]), vec(sc.local_box[1])
        self.origin, self.spacing = vec(vv.volume.origin), vec(vv.volume.spacing)
        self.rate = float(vv.volume.sampling_rate)
        self.step = float(min(vv.volume.spacing)) * self.rate
        self.last = vec(vv.volume.dims) - 1.0
        self.iso = [float(f32(x)) for x in vv.isovalues]
        self.dvr = vv.volume_render
        x = np.arange(256) / 255.0
        cm, om = vv.colormap.astype(np.float64), vv.opacitymap.astype(np.float64)
        self.colors = torch.from_numpy(np.stack([np.interp(x, cm[:, 0], cm[:, k]) for k in (1, 2, 3)], 1)).cuda()
        self.opacities = torch.from_numpy(np.interp(x, om[:, 0], om[:, 1])).cuda()

    def sample(self, p):
        l = torch.minimum(((p - self.origin) / self.spacing).clamp_min(0.0), self.last)
        i = torch.minimum(l.floor(), self.last - 1.0)
        f, i = l - i, i.long()
        out = 0.0
        for c in range(8):
            o = [(c >> k) & 1 for k in range(3)]
            w = 1.0
            for k in range(3):
                w = w * (f[:, k] if o[k] else 1.0 - f[:, k])
            out = out + w * self.vox[i[:, 2] + o[2], i[:, 1] + o[1], i[:, 0] + o[0]]
        return out

    @staticmethod
    def look_up(table, v):
        x = v.clamp(0.0, 1.0) * 255.0
        i = x.floor().clamp_max(254.0)
        r, i = x - i, i.long()
        a, b = table[i], table[i + 1]
        return a + (r.unsqueeze(-1) if a.dim() > 1 else r) * (b - a)

    def clip(self, org, d):
        a, b = (self.lo - org) / d, (self.hi - org) / d
        return torch.minimum(a, b).max(-1).values, torch.maximum(a, b).min(-1).values

    def march(self, org, d, color, primary):
        """Marches every ray; returns its colour, the t it ends at and whether
        an isosurface ended it there (with the isovalue)."""
        n = len(org)
        t0, t1 = self.clip(org, d)
        t0 = t0.clamp_min(0.0)
        end, hit, value = t1.clone(), torch.zeros(n, dtype=torch.bool, device="cuda"), torch.zeros(n).cuda().double()
        if not (self.iso or self.dvr):
            return color, end, hit, value
        eps = self.eps * self.step
        at = torch.nonzero((t0 <= t1) & (t0 + eps <= t1)).squeeze(-1)
        t_last, t = t0[at], t0[at] + eps
        s_last = self.sample(org[at] + t_last[:, None] * d[at])
        while len(at):
            o, dd, stop = org[at], d[at], t1[at]
            s = self.sample(o + t[:, None] * dd)
            live = t_last >= eps
            nxt = torch.minimum(t + self.step, stop)
            ih = torch.zeros_like(live)
            th, vh = t.clone(), torch.zeros_like(t)
            for iso in self.iso:
                m = live & (((iso >= s_last) & (iso < s)) | ((iso <= s_last) & (iso > s)))
                th = torch.where(m, t_last + (iso - s_last) / (s - s_last) * (t - t_last), th)
                vh = torch.where(m, torch.full_like(vh, iso), vh)
                ih |= m
            if ih.any():
                s = torch.where(ih, self.sample(o + th[:, None] * dd), s)
                t = torch.where(ih, th, t)
            opaque = torch.zeros_like(ih)
            if self.dvr:
                v = 0.5 * (s_last + s)
                w = (self.look_up(self.opacities, v) / self.rate).clamp(0.0, 1.0) * live
                c = color[at]
                if primary:
                    aw = ((1.0 - c[:, 3]) * w)[:, None]
                    c = c + aw * torch.cat([self.look_up(self.colors, v), torch.ones_like(aw)], 1)
                else:
                    c = c * (1.0 - (t - t_last) / self.step * w)[:, None]
                color[at] = c
                opaque = (c[:, :3].min(-1).values >= 1.0) | (c[:, 3] > self.alpha)
            done = ih | opaque | ~(nxt > t)
            end[at] = torch.where(ih | opaque, t, end[at])
            hit[at] = ih
            value[at] = torch.where(ih, vh, value[at])
            go = ~done
            at, t_last, s_last, t = at[go], t[go], s[go], nxt[go]
        return color, end, hit, value

    def camera(self):
        cam = self.sc.cameras[0]
        eye, up = vec(f32(x) for x in cam.eye), vec(f32(x) for x in cam.up)
        d = unit(vec(f32(x) for x in cam.center) - eye)
        right = unit(torch.linalg.cross(d, up))
        up = unit(torch.linalg.cross(right, d))
        mid = eye + d / math.tan(math.pi * cam.aov / 360.0)
        scale = 2.0 / (min(cam.width, cam.height) - 1.0)
        y, x = torch.meshgrid(torch.arange(cam.height, device="cuda"), torch.arange(cam.width, device="cuda"), indexing="ij")
        fx = (x.reshape(-1).double() - (cam.width - 1) / 2.0) * scale
        fy = (y.reshape(-1).double() - (cam.height - 1) / 2.0) * scale
        rays = unit(mid + fx[:, None] * right + fy[:, None] * up - eye)
        org = eye.expand_as(rays)
        t0, t1 = self.clip(org, rays)
        px = torch.nonzero((t0 <= t1) & (t1 >= 0)).squeeze(-1)
        return px, org[px], rays[px]

    def image(self):
        cam, L = self.sc.cameras[0], scenes.resolve_lights(self.sc.lighting, self.sc.cameras[0])
        px, org, d = self.camera()
        fb = torch.zeros(cam.height * cam.width, 4, dtype=torch.float64, device="cuda")
        color, end, hit, value = self.march(org, d, torch.zeros(len(px), 4, dtype=torch.float64, device="cuda"), True)
        k = torch.nonzero(hit).squeeze(-1)
        p = org[k] + end[k, None] * d[k]
        s = self.sample(p)
        e = torch.eye(3, dtype=torch.float64, device="cuda") * self.spacing
        g = torch.stack([(self.sample(p + e[a]) - s) / self.spacing[a] for a in range(3)], 1)
        nrm = g / g.square().sum(-1, keepdim=True).clamp_min(1e-12).sqrt()
        nrm = torch.where(((d[k] * nrm).sum(-1, keepdim=True) > 0), -nrm, nrm)
        surf = self.look_up(self.colors, value[k])
        o = color[k, 3:4].clone()
        kd = float(L.Kd) / len(L.sources)
        lit = float(L.Ka) * (1 - o) * surf
        o2 = o + kd * (1 - o) * o
        sp = p + self.eps * nrm
        for src in L.sources:
            to = unit(vec(src) - p)
            dot = (nrm * to).sum(-1, keepdim=True).clamp_min(0.0)
            lit = lit + kd * (1 - o) * (1 - o) * dot * surf
            if L.shadows:
                to = unit(vec(src) - sp)
                dot = (nrm * to).sum(-1, keepdim=True).clamp_min(0.0)
                c = torch.cat([-(1 - o2) * kd * dot * surf, torch.zeros_like(o)], 1)
                c, _, blocked, _ = self.march(sp, to, c, False)
                fb.index_add_(0, px[k], torch.where(blocked[:, None], c, torch.zeros_like(c)))
        color[k, :3] += lit
        color[k, 3:4] = o2
        fb.index_add_(0, px, color)
        return fb.reshape(cam.height, cam.width, 4)
