"""The scene raycast's four-lane kernel where its deferred decisions could go wrong: coincident instances
(contenders past a lane's list, past a ray's row), rays it hands to the one-lane kernel, inverses that
are not the matrices', grazing rays. The answer is that of the batched launch on every (ray, instance) pair."""
import numpy as np
import pytest

import mbvh_amd as M
from mbvh_amd import geometry as G, workloads as W
from helpers import build_mesh
from test_gpu_scene import GEOMS, _pairwise, _same
from test_gpu_scene_points import _roots

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = M.Context(0)
    yield c
    c.close()


@pytest.fixture(scope="module")
def meshes(ctx):
    built = [build_mesh(f()) for f in GEOMS]
    ms = [ctx.upload(t, g.positions, idx) for g, idx, t in built]
    yield [b[0] for b in built], ms
    for m in ms:
        m.free()


def _check(ctx, ms, w, **kw):
    sc = ctx.scene(ms, w.matrix_world, w.matrix_world_inverse, w.instance_geometry)
    got = sc.raycast_first(w.origins, w.directions, **kw)
    ref = _pairwise(ctx, ms, w, None, **kw)
    _same(got, ref)
    sc.free()
    return ref


@pytest.mark.parametrize("copies", [2, 4, 5, 7, 40])
def test_coincident_instances(ctx, meshes, copies):
    geos, ms = meshes
    w = W.scene_rays(geos, 3 * copies, 1500, seed=21)
    for k in range(3 * copies):
        for a in (w.matrix_world, w.matrix_world_inverse, w.instance_geometry):
            a[k] = a[k // copies * copies]
    ref = _check(ctx, ms, w)
    hit = ref["instance"] != M.NO_HIT
    assert hit.any() and np.all(ref["instance"][hit] % copies == 0)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 1000])
def test_ray_counts(ctx, meshes, n):
    geos, ms = meshes
    _check(ctx, ms, W.scene_rays(geos, 9, n, seed=22))


@pytest.mark.parametrize("kind", ["axis", "mixed", "unrotated"])
def test_zero_direction_components(ctx, meshes, kind):
    geos, ms = meshes
    w = W.scene_rays(geos, 16, 1200, seed=23)
    if kind == "unrotated":  # zero components only after the instance's transform
        for k in range(16):
            m = np.eye(4)
            m[:3, 3] = w.matrix_world[k].reshape(4, 4).T[:3, 3]
            w.matrix_world[k] = m.T.reshape(-1)
            w.matrix_world_inverse[k] = np.linalg.inv(m).T.reshape(-1)
    rows = slice(None) if kind == "axis" else slice(0, None, 3)
    w.directions[rows] = np.eye(3, dtype=np.float32)[np.arange(1200) % 3][rows]
    ctr = w.matrix_world.reshape(-1, 4, 4)[np.arange(1200) % 16, 3, :3]
    w.origins[rows] = (ctr + 0.1 - 60 * w.directions)[rows]
    assert (_check(ctx, ms, w)["face"][rows] != M.NO_HIT).any()


@pytest.mark.parametrize("two", [False, True])
@pytest.mark.parametrize("side", [M.FRONT_SIDE, M.DOUBLE_SIDE])
def test_rays_along_box_planes(ctx, two, side):
    """Rays parallel to one or two axes from whole coordinates, where the boxes of unrotated instances begin as
    well: the reference's split-plane shortcut then skips children that may hold the nearer hit."""
    rng = np.random.default_rng(27)
    at = rng.integers(-6, 7, (400, 3)).astype(float)
    axis = rng.integers(0, 3, 400)
    quads = np.repeat(at[:, None], 4, 1)
    u, v = np.eye(3)[(axis + 1) % 3], np.eye(3)[(axis + 2) % 3]
    quads[:, 1] += u
    quads[:, 2] += u + v
    quads[:, 3] += v
    f = np.arange(400)[:, None] * 4
    g, idx, tree = build_mesh(G.Geometry(quads.reshape(-1, 3).astype(np.float32),
                                         np.concatenate([f, f + 1, f + 2, f, f + 2, f + 3], 1).reshape(-1).astype(np.uint32)),
                              leaf=1)
    ms = [ctx.upload(tree, g.positions, idx)]
    w = W.scene_rays([g], 4, 4000, seed=28)
    for k in range(4):
        m = np.eye(4)
        m[:3, 3] = rng.integers(-9, 10, 3)
        w.matrix_world[k] = m.T.reshape(-1)
        w.matrix_world_inverse[k] = np.linalg.inv(m).T.reshape(-1)
    d = rng.choice([-1.0, 1.0], (4000, 3)) * (1.0 if two else rng.uniform(0.2, 1.0, (4000, 3)))
    zero = rng.integers(0, 3, 4000)
    d[np.arange(4000), zero] = np.where(rng.random(4000) < 0.5, 0.0, -0.0)
    if two:
        d[np.arange(4000), (zero + 1) % 3] = 0.0
    w.directions[:] = d / np.linalg.norm(d, axis=1, keepdims=True)
    w.origins[:] = rng.integers(-12, 13, (4000, 3))
    ref = _check(ctx, ms, w, side=side)
    assert (ref["face"] != M.NO_HIT).sum() > 500
    ms[0].free()


@pytest.mark.parametrize("kind", ["shifted", "scaled", "projective", "sheared"])
def test_any_inverse(ctx, meshes, kind):
    geos, ms = meshes
    w = W.scene_rays(geos, 12, 1500, seed=24, non_uniform=0.5)
    inv = w.matrix_world_inverse
    if kind == "shifted":
        inv[:, 12:15] += 0.05
    elif kind == "scaled":
        inv[:, :15] *= np.float32(1.25)
    elif kind == "projective":
        inv[:, 15] = 1.0 + 1e-3
        inv[:, 3] = 1e-4
    else:
        for k in range(12):
            m = w.matrix_world[k].reshape(4, 4).T.astype(np.float64)
            m[:3, :3] = m[:3, :3] @ np.array([[1, 0.9, 0], [0, 1, 0.4], [0, 0, 1]])
            w.matrix_world[k] = m.T.reshape(-1)
            inv[k] = np.linalg.inv(w.matrix_world[k].reshape(4, 4).astype(np.float64)).reshape(-1)
    _check(ctx, ms, w, side=M.DOUBLE_SIDE)


def test_grazing_rays(ctx):
    """Rays in the plane of whole rows of triangles: undecided hits by the dozen."""
    grid = np.arange(17, dtype=np.float32) / 4
    x, y = np.meshgrid(grid, grid, indexing="ij")
    pos = np.stack([x, y, 0 * x], -1).reshape(-1, 3)
    a = (np.arange(16)[:, None] * 17 + np.arange(16)[None, :]).reshape(-1)
    g0 = G.Geometry(pos, np.stack([a, a + 1, a + 17, a + 1, a + 18, a + 17], -1).reshape(-1).astype(np.uint16))
    g, idx, tree = build_mesh(g0)
    ms = [ctx.upload(tree, g.positions, idx)]
    w = W.scene_rays([g], 6, 1024, seed=25)
    rng = np.random.default_rng(26)
    k = rng.integers(0, 6, 1024)
    m = w.matrix_world.reshape(-1, 4, 4)[k].transpose(0, 2, 1).astype(np.float64)
    p = np.concatenate([rng.uniform(0, 4, (1024, 2)), np.zeros((1024, 1))], 1)
    q = np.concatenate([rng.uniform(-9, -5, (1024, 2)), 1e-6 * rng.standard_normal((1024, 1))], 1)
    p, q = (np.einsum("nij,nj->ni", m[:, :3, :3], v) + m[:, :3, 3] for v in (p, q))
    w.origins[:] = q
    d = p - w.origins.astype(np.float64)
    w.directions[:] = d / np.linalg.norm(d, axis=1, keepdims=True)
    _check(ctx, ms, w, side=M.DOUBLE_SIDE)
    ms[0].free()


@pytest.mark.parametrize("kind,count,n", [("random", 3, (1 << 18) + 37), ("camera", 3, (1 << 18) + 37), ("camera", 1, 140000),
                                          ("random", 3, (1 << 20) + 1237), ("camera", 3, (1 << 20) + 300000),
                                          ("within", 33, (1 << 18) + 37)])
def test_many_rays(ctx, meshes, kind, count, n):
    """Calls large enough to be sampled for coherence (a camera's rows of rays are coherent and go to one lane per
    ray, from within the scene also at a wider spread), for one instance to do without, and to be cut: a second
    part below and above the sampled size."""
    geos, ms = meshes
    w = W.scene_rays(geos, count, n, seed=29)
    if kind != "random":
        k = np.arange(n) / n
        at = w.matrix_world.reshape(-1, 4, 4)[:, 3, :3]
        ctr, half = at.mean(0), np.abs(at - at.mean(0)).max() + 1.5
        eye = ctr + half * np.array([0.5, 4.0, 0.3] if kind == "camera" else [0.1, 0.6, 0.1])
        at = ctr + half * np.stack([2 * (1000 * k % 1) - 1, 0 * k, 2 * k - 1], 1)
        w.origins[:] = eye
        w.directions[:] = (at - eye) / np.linalg.norm(at - eye, axis=1, keepdims=True)
    ref = _check(ctx, ms, w)
    assert (ref["face"] != M.NO_HIT).sum() > n // 100


def test_several_roots(ctx, meshes):
    """Instances of a mesh of four roots among others."""
    geos, ms = meshes
    g = G.torus_knot(0.8, 0.25, 90, 9, 2, 3).ensure_index()
    g, idx, tree = build_mesh(g, ranges=_roots(g, 4))
    assert len(tree.roots) == 4
    mesh = ctx.upload(tree, g.positions, idx)
    ref = _check(ctx, [mesh, ms[0]], W.scene_rays([g, geos[0]], 9, 2000, seed=30))
    assert (ref["face"] != M.NO_HIT).any()
    mesh.free()
