"""The FP32 triangle frames behind the closest-point kernels (four lanes per query, packets of 64):
where their bounds could go wrong, the answers must still be the FP64 oracle's and the widths agree."""
import numpy as np
import pytest

import mbvh_amd as M
from mbvh_amd import geometry as G
import oracle_py as O
from helpers import build_mesh, check_closest_parity

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = M.Context(0)
    yield c
    c.close()


def _geo(tris):
    pos = np.asarray(tris, np.float64).astype(np.float32).reshape(-1, 3)
    return G.Geometry(pos, np.arange(pos.shape[0], dtype=np.uint32))


def _soup(rng, n, size, spread, thin):
    a = rng.uniform(-spread, spread, (n, 3))
    e = rng.standard_normal((n, 3)) * size
    return np.stack([a, a + e, a + e * rng.uniform(-0.5, 1.5, (n, 1)) + rng.standard_normal((n, 3)) * size * thin], 1)


def collinear(n):
    """n exactly collinear triangles (corners a, a + e, a + 2 e in any order, whole numbers) 16 apart, a
    triangle at least 1.25 from each one's middle, and queries within 0.5 of the middles: (triangles, queries,
    distances). All products are exact in FP32, so the exact step has no noise either."""
    rng = np.random.default_rng(32)
    side = int(np.ceil(n ** (1 / 3)))
    mid = 16.0 * np.stack(np.unravel_index(np.arange(n), (side,) * 3), 1)
    e = rng.integers(-3, 4, (n, 3)).astype(float)
    e[:, 0] = 1 + rng.integers(0, 3, n)
    line = np.stack([mid - e, mid, mid + e], 1)
    line = np.stack([x[rng.permutation(3)] for x in line])
    axis = rng.integers(0, 3, n)
    other = mid[:, None, :] + rng.integers(-2, 3, (n, 3, 3))
    other[np.arange(n), 0, (axis + 1) % 3] += 4
    other[np.arange(n), 1, (axis + 2) % 3] += 4
    other[np.arange(n), :, axis] = mid[np.arange(n), axis][:, None] + 1.5
    off = 0.25 * rng.integers(-1, 2, (n, 3))
    t = np.clip((off * e).sum(1) / (e * e).sum(1), -1, 1)
    return np.concatenate([line, other]), mid + off, np.linalg.norm(off - t[:, None] * e, axis=1)


def segments(order, n=3000):
    """Strands of n segments stored as triangles with two equal corners ("abb", "aba" or "aab")."""
    rng = np.random.default_rng(33)
    p = np.cumsum(np.concatenate([rng.uniform(-2, 2, (n // 100, 1, 3)), 0.1 * rng.standard_normal((n // 100, 100, 3))], 1), 1)
    ends = dict(a=p[:, :-1].reshape(-1, 3), b=p[:, 1:].reshape(-1, 3))
    return np.stack([ends[c] for c in order], 1).astype(np.float32)


def _cases(name):
    if name == "line":
        return collinear(1000)[:2]
    if name == "lines":  # none of the triangles bounds the search
        tris, q, _ = collinear(1000)
        return tris[:1000], q
    if name in ("abb", "aba", "aab"):
        return segments(name), np.random.default_rng(34).uniform(-3, 3, (4099, 3))
    rng = np.random.default_rng(31)
    if name.startswith("few"):  # a leaf alone: odd and even counts of the two-triangle step
        t = _soup(rng, int(name[3:]), 1.0, 2.0, 1.0)
        return t, rng.uniform(-4, 4, (130, 3))
    if name == "thin":  # heights down to 1e-7 of the length, and degenerate triangles among them
        t = np.concatenate([_soup(rng, 400, 0.5, 2.0, 10.0 ** -k) for k in range(0, 8)])
        flat = _soup(rng, 90, 0.5, 2.0, 1.0)
        flat[:30, 1] = flat[:30, 0]                       # two equal corners
        flat[30:60, 2] = 0.5 * (flat[30:60, 0] + flat[30:60, 1])  # collinear up to the corners' rounding
        flat[60:, 1:] = flat[60:, :1]                     # a point
        return np.concatenate([t, flat]), rng.uniform(-3, 3, (4099, 3))
    if name == "fan":  # the closest feature of every query above the tip is the vertex all 96 share
        w = np.arange(97) / 96 * 2 * np.pi
        ring = np.stack([np.cos(w), np.sin(w), -1.5 + 0 * w], 1)
        t = np.stack([np.zeros((96, 3)), ring[:-1], ring[1:]], 1)
        q = np.stack([rng.uniform(-0.1, 0.1, 300), rng.uniform(-0.1, 0.1, 300), rng.uniform(0.5, 3, 300)], 1)
        return t, np.concatenate([q, rng.uniform(-2, 2, (300, 3))])
    if name == "twice":  # every triangle there twice: exact ties everywhere
        t = _soup(rng, 700, 0.3, 2.0, 1.0)
        return np.concatenate([t, t]), rng.uniform(-3, 3, (1500, 3))
    if name == "far":  # small triangles seen from 10^5 of their sizes
        t = _soup(rng, 3000, 1e-3, 1.0, 1.0)
        return t, rng.standard_normal((700, 3)) * 100.0
    if name == "on":  # queries on the triangles: corners, edges, insides
        t = _soup(rng, 1200, 0.4, 2.0, 1.0)
        t32 = t.astype(np.float32).astype(np.float64)
        w = rng.dirichlet([1, 1, 1], 1200)
        w[:300] = np.eye(3)[rng.integers(0, 3, 300)]
        w[300:600, 2] = 0
        w[300:600] /= w[300:600].sum(1, keepdims=True)
        return t, (w[:, :, None] * t32).sum(1)
    raise KeyError(name)


@pytest.mark.parametrize("name", ["few1", "few2", "few3", "few9", "few11", "thin", "fan", "twice", "far", "on", "line", "lines", "abb", "aba", "aab"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("max_t", [float("inf"), 0.7])
def test_frames(ctx, name, dtype, max_t):
    tris, q = _cases(name)
    q = q.astype(dtype)
    g, idx, tree = build_mesh(_geo(tris))
    om = O.OracleMesh(g.positions, idx, tree.roots)
    ref = om.closest_point(q, 0.0, max_t)
    got = {}
    for lanes in (4, 64):
        ctx.set_point_lanes(lanes)
        mesh = ctx.upload(tree, g.positions, idx)
        got[lanes] = mesh.closest_point(q, 0.0, max_t)
        mesh.free()
        print(name, lanes, check_closest_parity(om, q, got[lanes], ref, f"{name} {lanes}"), flush=True)
    ctx.set_point_lanes(0)
    for k in got[4]:
        assert np.array_equal(got[4][k].view(np.uint32), got[64][k].view(np.uint32)), k


def test_frames_follow_a_refit(ctx):
    """A refit rewrites the frames: the answers are those of a mesh uploaded with the new positions."""
    tris, q = _cases("thin")
    g, idx, tree = build_mesh(_geo(tris))
    moved = (g.positions.reshape(-1, 3) * np.float32(1.25) + np.float32(0.1)).astype(np.float32)
    q = q.astype(np.float32)
    mesh = ctx.upload(tree, g.positions, idx)
    roots = mesh.refit(moved)
    fresh = ctx.upload(M.Tree(roots, None), moved, idx)
    for lanes in (4, 64):
        ctx.set_point_lanes(lanes)
        a, b = mesh.closest_point(q), fresh.closest_point(q)
        for k in a:
            assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), (lanes, k)
    ctx.set_point_lanes(0)
    mesh.free()
    fresh.free()
