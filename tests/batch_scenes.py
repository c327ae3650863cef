"""Small datasets for the batched and served tests: two smooth seeded
volumes over the unit cube (compositing, iso 0.5) and two blob meshes."""
import numpy as np

from galaxy_amd import abi, scenes, workloads

f32 = np.float32


def smooth_volume(n, seed):
    """n^3 voxels of a smooth seeded field in [0, 1] over the unit cube."""
    rng = np.random.default_rng(seed)
    x = np.linspace(0, 1, n, dtype=np.float64)
    Z, Y, X = np.meshgrid(x, x, x, indexing="ij")
    f = np.zeros_like(X)
    for k in range(4):
        a = rng.normal(size=3)
        f += np.sin(2.5 * (k + 1) * (a[0] * X + a[1] * Y + a[2] * Z) + rng.uniform(0, 6.3)) / (k + 1)
    f = (f - f.min()) / (f.max() - f.min())
    delta = f32(1.0 / (n - 1))
    return scenes.VolumeDesc(f.astype(f32), (f32(0),) * 3, (delta,) * 3, sampling_rate=0.5,
                             local_box=workloads.UNIT_BOX, global_box=workloads.UNIT_BOX)


def dataset_descs():
    d = np.linspace(0.0, 1.0, 8)
    rgb, op = workloads.VOLUME_RENDER_TF
    out = []
    for k, n in enumerate((40, 56)):
        vol = smooth_volume(n, 10 + k)
        vv = scenes.VolumeVisDesc(vol, colormap=np.c_[d, rgb].astype(f32), opacitymap=np.c_[d, 4 * op].astype(f32),
                                  isovalues=np.array([0.5], f32), volume_render=True)
        out.append(scenes.SceneDesc(volume_vis=[vv], local_box=workloads.UNIT_BOX, global_box=workloads.UNIT_BOX))
    out.append(workloads.blob_scene(3000, 7))
    out.append(workloads.blob_scene(20000, 8))
    return out


def graded_scene(seed, levels=34, per=12):
    """Small triangles around the corners of cubes that halve from level to
    level towards the origin: a deep tree over few primitives."""
    rng = np.random.default_rng(seed)
    x = 0.5 ** np.repeat(np.arange(levels), per)
    c = x[:, None] * rng.choice([0.25, 1.0], (len(x), 3))
    v = c[:, None] + 0.1 * x[:, None, None] * rng.uniform(-0.5, 0.5, (len(x), 3, 3))
    box = ((-4.0,) * 3, (4.0,) * 3)
    return scenes.SceneDesc(meshes=[scenes.MeshDesc(v.reshape(-1, 3).astype(f32),
                                                    np.arange(3 * len(x), dtype=np.uint32).reshape(-1, 3))],
                            local_box=box, global_box=box)


def rays_at_triangles(sc, n, seed):
    """Origins around the scene, directions to random triangles of its mesh."""
    rng = np.random.default_rng(seed)
    m = sc.meshes[0]
    c = m.vertices[m.indices].astype(float).mean(1)
    o = rng.uniform(-1.0, 2.0, (n, 3))
    d = c[rng.integers(len(c), size=n)] - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return abi.HostRays.from_arrays(o.astype(f32), d.astype(f32), np.zeros(n, f32), np.full(n, 1e30, f32))
