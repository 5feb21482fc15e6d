"""The scene closest point's FP32 walk (instances placed by similarities) where its bounds and lists could
go wrong: ties between many triangles and instances, points its lists cannot hold, far, tiny and
non-finite queries, large and small scales. The answer is the one-lane kernel's, which measures in
double as it walks, bit for bit."""
import numpy as np
import pytest

import mbvh_amd as M
from mbvh_amd import geometry as G
from helpers import build_mesh
from test_gpu_closest_frames import collinear, segments

pytestmark = pytest.mark.gpu

GEOMS = [lambda: G.sphere(1.0, 60, 40), lambda: G.torus_knot(0.8, 0.25, 90, 9, 2, 3), lambda: G.sphere(0.7, 3, 2)]


@pytest.fixture(scope="module")
def setup():
    ctx = M.Context(0)
    built = [build_mesh(f()) for f in GEOMS]
    meshes = [ctx.upload(t, g.positions, idx) for g, idx, t in built]
    yield ctx, meshes
    for m in meshes:
        m.free()
    ctx.close()


def matrices(count, rng, scale=(0.5, 2.0), span=6.0, stretch=1.0):
    q = rng.normal(size=(count, 4))
    x, y, z, w = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    r = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                  2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                  2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], axis=1).reshape(-1, 3, 3)
    m = np.zeros((count, 4, 4))
    m[:, :3, :3] = r * rng.uniform(*scale, size=(count, 1, 1)) * np.array([1.0, 1.0, stretch])
    m[:, :3, 3] = rng.uniform(-span, span, size=(count, 3))
    m[:, 3, 3] = 1
    return m


LEAST = 200000


def check(setup, m, which, points, fill_scale=1.0):
    ctx, meshes = setup
    world = np.ascontiguousarray(m.transpose(0, 2, 1).reshape(-1, 16), dtype=np.float32)
    inverse = np.linalg.inv(world.reshape(-1, 4, 4).astype(np.float64)).reshape(-1, 16).astype(np.float32)
    sc = ctx.scene(meshes, world, inverse, np.asarray(which, dtype=np.uint32))
    # the walk takes 200,000 points or more: others around the scene bring them there
    fill = np.random.default_rng(0).uniform(-8, 8, size=(LEAST, 3)) * fill_scale
    points = np.ascontiguousarray(np.concatenate([points, fill]), dtype=np.float32)
    got = sc.closest_point(points)
    ctx.set_point_lanes(1)
    ref = sc.closest_point(points)
    ctx.set_point_lanes(0)
    sc.free()
    for k in ref:
        np.testing.assert_array_equal(got[k].view(np.uint32), ref[k].view(np.uint32), err_msg=k)
    return {k: v[:len(points) - LEAST] for k, v in ref.items()}


@pytest.mark.parametrize("n", [1, 17, 65, 3001])
@pytest.mark.parametrize("count", [1, 2, 40])
def test_counts(setup, n, count):
    rng = np.random.default_rng(n + count)
    ref = check(setup, matrices(count, rng), rng.integers(0, 3, count), rng.uniform(-7, 7, size=(n, 3)))
    assert np.all(ref["face"] != M.NO_HIT)


@pytest.mark.parametrize("copies,n", [(2, 2000), (40, 2000)])
def test_coincident_instances(setup, copies, n):
    """Every triangle ties with its copies: past a row, past a lane's list, more such points than a wave each."""
    rng = np.random.default_rng(copies)
    m = np.repeat(matrices(2, rng), copies, axis=0)
    ref = check(setup, m, np.repeat([0, 1], copies), rng.uniform(-5, 5, size=(n, 3)))
    assert np.all(ref["instance"] % copies == 0)


@pytest.mark.parametrize("spread", [0.0, 1e-4])
def test_long_walks(setup, spread):
    """Points at the centres of spheres, on their poles and axes, and on vertices."""
    rng = np.random.default_rng(3)
    m = matrices(6, rng)
    local = np.concatenate([np.zeros((60, 3)), np.tile([[0, 1, 0], [0, -1, 0], [0, 3, 0], [0, 0.2, 0]], (60, 1)),
                            G.sphere(1.0, 60, 40).positions.reshape(-1, 3)[:200]]) + spread * rng.normal(size=(500, 3))
    at = rng.integers(0, 6, 500)
    check(setup, m, [0] * 6, np.einsum("nij,nj->ni", m[at][:, :3, :3], local) + m[at][:, :3, 3])


@pytest.mark.parametrize("size", [1e3, 1e6, 1e15, 3e19, 1e-10])
def test_far_and_tiny(setup, size):
    rng = np.random.default_rng(5)
    check(setup, matrices(5, rng), [0, 1, 2, 0, 1], size * rng.normal(size=(300, 3)))


@pytest.mark.parametrize("scale,span", [((1e-5, 1e-4), 1e-3), ((1e4, 1e5), 1e5), ((1e-3, 1e3), 50.0), ((1.0, 1.0), 1e4)])
def test_scales(setup, scale, span):
    rng = np.random.default_rng(6)
    check(setup, matrices(12, rng, scale, span), rng.integers(0, 3, 12), span * rng.uniform(-1.2, 1.2, size=(2000, 3)), span / 6)


@pytest.mark.parametrize("stretch", [1.0 + 1e-7, 1.0 + 1e-5, 1.0 + 1e-4, 1.5, -1.0])
def test_stretched(setup, stretch):
    """Either side of the similarity rule, and mirrored."""
    rng = np.random.default_rng(7)
    check(setup, matrices(12, rng, stretch=stretch), rng.integers(0, 3, 12), rng.uniform(-7, 7, size=(2000, 3)))


def test_not_finite(setup):
    rng = np.random.default_rng(8)
    p = rng.uniform(-7, 7, size=(64, 3))
    p[0::8, 0], p[1::8, 1], p[2::8] = np.nan, np.inf, -np.inf
    ref = check(setup, matrices(3, rng), [0, 1, 2], p)
    assert np.all(ref["face"][0::8] == M.NO_HIT) and np.all(ref["face"][3::8] != M.NO_HIT)


def test_collinear(setup):
    """Exactly collinear triangles are the nearest (moved by whole numbers and doubled, so still exactly so)."""
    ctx, _ = setup
    tris, local, dist = collinear(1000)
    pos = tris.astype(np.float32).reshape(-1, 3)
    g, idx, tree = build_mesh(G.Geometry(pos, np.arange(len(pos), dtype=np.uint32)))
    mesh = ctx.upload(tree, g.positions, idx)
    m = np.stack([np.eye(4), np.diag([2.0, 2.0, 2.0, 1.0])])
    m[1, :3, 3] = 512
    world = np.ascontiguousarray(m.transpose(0, 2, 1).reshape(-1, 16), dtype=np.float32)
    inverse = np.linalg.inv(world.reshape(-1, 4, 4).astype(np.float64)).reshape(-1, 16).astype(np.float32)
    sc = ctx.scene([mesh], world, inverse, np.zeros(2, np.uint32))
    points = np.concatenate([local, 2 * local + 512]).astype(np.float32)
    got = sc.closest_point(np.tile(points, (LEAST // len(points), 1)))
    want = np.tile(np.concatenate([dist, 2 * dist]), LEAST // len(points))
    np.testing.assert_allclose(got["distance"], want, rtol=1e-6)
    assert np.array_equal(got["instance"], np.tile(np.repeat([0, 1], 1000), LEAST // len(points)))
    sc.free()
    mesh.free()


@pytest.mark.parametrize("corners", ["abb", "aba", "aab"])
def test_segments(setup, corners):
    """Instances whose triangles all have two equal corners. Where those are a, a, b the closest point only
    exists for points that a is nearest to (elsewhere it is 0 / 0), and no triangle bounds the walk."""
    ctx, _ = setup
    tris = segments(corners, 300)
    pos = tris.reshape(-1, 3)
    g, idx, tree = build_mesh(G.Geometry(pos, np.arange(len(pos), dtype=np.uint32)))
    mesh = ctx.upload(tree, g.positions, idx)
    rng = np.random.default_rng(9)
    m = matrices(3, rng, span=3.0)
    world = np.ascontiguousarray(m.transpose(0, 2, 1).reshape(-1, 16), dtype=np.float32)
    inverse = np.linalg.inv(world.reshape(-1, 4, 4).astype(np.float64)).reshape(-1, 16).astype(np.float32)
    sc = ctx.scene([mesh], world, inverse, np.zeros(3, np.uint32))
    q = rng.uniform(-6, 6, (2000, 3)).astype(np.float32)
    got = sc.closest_point(np.tile(q, (LEAST // 2000, 1)))
    w = world.reshape(3, 4, 4).astype(np.float64)
    a, b = (np.concatenate([tris[:, corners.index(c)].astype(np.float64) @ x[:3, :3] + x[3, :3] for x in w]) for c in "ab")
    e = b - a
    t = ((q.astype(np.float64) @ e.T) - (a * e).sum(1)) / (e * e).sum(1)
    d = np.linalg.norm(q[:, None] - a - np.clip(t, 0, 1)[:, :, None] * e, axis=2)
    if corners == "aab":
        d[t > 0] = np.inf
    np.testing.assert_allclose(got["distance"], np.tile(d.min(1), LEAST // 2000), rtol=1e-6)
    sc.free()
    mesh.free()


def _roots(g, parts):
    """The geometry's triangles in `parts` ranges, a root each."""
    edges = np.linspace(0, g.index.size // 3, parts + 1).astype(int)
    return [(int(a), int(b - a)) for a, b in zip(edges[:-1], edges[1:])]


def test_several_roots(setup):
    """Instances of a mesh of four roots among others."""
    ctx, meshes = setup
    g = G.torus_knot(0.8, 0.25, 90, 9, 2, 3).ensure_index()
    g, idx, tree = build_mesh(g, ranges=_roots(g, 4))
    assert len(tree.roots) == 4
    mesh = ctx.upload(tree, g.positions, idx)
    rng = np.random.default_rng(10)
    check((ctx, [mesh, meshes[0]]), matrices(9, rng), np.arange(9) % 2, rng.uniform(-7, 7, size=(3000, 3)))
    mesh.free()


def test_second_part(setup):
    """More points than a launch takes, in the caller's visit order (outputs in place) and without one (the
    second part's buffers moved)."""
    import torch

    ctx, meshes = setup
    rng = np.random.default_rng(11)
    m = matrices(5, rng)
    world = np.ascontiguousarray(m.transpose(0, 2, 1).reshape(-1, 16), dtype=np.float32)
    inverse = np.linalg.inv(world.reshape(-1, 4, 4).astype(np.float64)).reshape(-1, 16).astype(np.float32)
    sc = ctx.scene(meshes, world, inverse, np.arange(5, dtype=np.uint32) % 3)
    n = (1 << 20) + 4321
    q = rng.uniform(-8, 8, (n, 3)).astype(np.float32)
    ctx.set_point_lanes(1)
    ref = sc.closest_point(q)
    ctx.set_point_lanes(0)
    points = torch.as_tensor(q, device="cuda")
    order = torch.as_tensor(rng.permutation(n).astype(np.uint32).view(np.int32), device="cuda")
    for visit in (0, order.data_ptr()):
        out = {k: torch.full((n, 3) if k in ("point", "barycoord") else (n,), -7, dtype=torch.int32, device="cuda")
               for k in ("face", "instance", "distance", "point", "barycoord")}
        torch.cuda.synchronize()
        sc.closest_point_d(points.data_ptr(), n, *[out[k].data_ptr() for k in out], order_ptr=visit)
        ctx.synchronize()
        for k in ref:
            np.testing.assert_array_equal(out[k].cpu().numpy(), ref[k].view(np.int32), err_msg=k)
    sc.free()
