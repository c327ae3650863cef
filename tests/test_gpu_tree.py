"""The restructuring of the BVH build where its result is known: seven primitives
and one far away.  The seven are one treelet below the root, so the built tree
has to be the cheapest of all binary trees over the eight (any subtree a leaf,
the root not).  (Trees over fewer than eight primitives are not restructured.)"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
f32 = np.float32
CI = 1.2   # cost of visiting a node


@pytest.fixture(scope="module")
def hip():
    from galaxy_amd import lib as glib
    return glib.HipBackend()


def _triangles(kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "lattice":   # equal boxes in a row and a plane: many splits of equal cost
        at = np.array([[k % 4, k // 4 * (seed % 2), 0] for k in range(7)], float)
        return (at[:, None] + np.array([[0, 0, 0], [0.5, 0, 0], [0, 0.5, 0.25]])).astype(f32)
    size = {"small": 0.05, "large": 1.0, "mixed": 10.0 ** rng.uniform(-3, 0, (7, 1, 1))}[kind]
    return (rng.uniform(0, 1, (7, 1, 3)) + size * rng.uniform(-0.5, 0.5, (7, 3, 3))).astype(f32)


def _far(v):
    """A triangle beyond the middle of the scene in x, where the first split falls."""
    return (np.array([[[0, 0.4, 0.4], [0.1, 0.4, 0.4], [0, 0.5, 0.5]]]) + [40 * v[..., 0].max(), 0, 0]).astype(f32)


def _cheapest(v, ct):
    """SAH cost of the cheapest tree over the triangles' boxes, relative to the root's surface."""
    lo, hi = v.min(1).astype(float), v.max(1).astype(float)
    n = len(v)
    best, area = np.zeros(1 << n), np.zeros(1 << n)
    for s in range(1, 1 << n):
        m = [j for j in range(n) if s >> j & 1]
        d = hi[m].max(0) - lo[m].min(0)
        area[s] = d[0] * d[1] + d[1] * d[2] + d[2] * d[0]
        inner, q = np.inf, (s - 1) & s
        while q:
            inner = min(inner, CI * area[s] + best[q] + best[s ^ q])
            q = (q - 1) & s
        best[s] = min(inner, ct * area[s] * len(m)) if s != (1 << n) - 1 else inner
    # the far primitive alone on one side of the root: the tree the build can reach
    assert np.isclose(best[-1], CI * area[-1] + best[(1 << n) // 2 - 1] + best[(1 << n) // 2], rtol=1e-12)
    return best[-1] / area[-1]


@pytest.mark.parametrize("kind", ["small", "large", "mixed", "lattice"])
def test_seven_primitives_give_the_cheapest_tree(hip, kind):
    L = hip.L
    ct = L.gxy_get_bvh_prim_cost(0)
    for seed in range(12):
        v = _triangles(kind, seed)
        v = np.concatenate([v, _far(v)])
        m = hip.model_create()
        hip.model_add_triangles(m, v.reshape(-1), np.arange(24, dtype=np.uint32), None, None, None)
        hip.model_commit(m)
        nodes, leaves, depth, sah = C.c_int(), C.c_int(), C.c_int(), C.c_float()
        assert L.gxy_model_bvh_stats(m, C.byref(nodes), C.byref(leaves), C.byref(depth), C.byref(sah)) == 0
        assert L.gxy_model_destroy(m) == 0
        # a tree within 1e-5 of the cheapest is left as it is; sums of 15 terms in float
        want = _cheapest(v, ct)
        assert abs(sah.value - want) <= 3e-5 * want, (seed, sah.value, want)
