"""The work a program has this engine do, as cases that can be timed and compared.

Every case is one call, or one step of a program's loop, through the public entry points of
`mbvh_amd`: first-hit and all-hits raycasts, closest points, their backward passes after a refit,
instanced meshes and scenes, and the device build. Queries and outputs are resident in HBM, except
in the host case, whose arrays a JavaScript or numpy caller holds in host memory.

Meshes are named by their generator: "knot" is TorusKnot(10, 3, a, b) with 2ab triangles, "ico" the
noise-displaced Icosahedron(1, a) with 20 (a + 1)^2 triangles. `instances` of `meshes` different
geometries (torus knots and spheres, triangle counts log-uniform) make the instanced cases.
"""
from __future__ import annotations

import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "three-mesh-bvh_amd",
                                "python"))
import mbvh_amd as M  # noqa: E402  (after torch: both use one HIP runtime)
from mbvh_amd import geometry as G  # noqa: E402

INF = float("inf")
PAIR_LIMIT = 8_000_000_000  # (query, triangle) pairs that exact() tries one by one


def listed():
    return [
        # A few picking or visibility rays against one model: what an interactive program sends per
        # frame. The time is launches and the longest chain of dependent reads.
        dict(name="ray_1k", kind="ray", mesh="knot", a=400, b=100, n=1000, side="front", dtype="f32"),
        # A 256 x 256 image or sensor sweep of rays from around an 80k-triangle model.
        dict(name="ray_65k", kind="ray", mesh="knot", a=400, b=100, n=65536, side="front", dtype="f32"),
        # One step of a loop that fits a mesh to ray measurements: refit the tree to the moved
        # vertices, first hits, gradients with respect to rays and vertices (deterministic sums).
        dict(name="ray_train_1m", kind="ray_train", mesh="ico", a=200, b=0, n=1 << 20),
        # Every hit along each ray, both sides: thickness, inside / outside and volume sampling.
        dict(name="ray_all_262k", kind="ray_all", mesh="knot", a=400, b=100, n=262144, side="double"),
        # The drop-in host path: double-precision points in host arrays, results back in host arrays.
        dict(name="point_host_f64_30k", kind="point_host", mesh="knot", a=400, b=100, n=30001, dtype="f64"),
        # A distance field sampled on a grid, ordered in the call, in packets of 64 (coherent points).
        dict(name="point_grid_128", kind="point", mesh="knot", a=800, b=200, n=128 ** 3, grid=128, lanes=64,
             dtype="f32"),
        # A scattered point cloud around the same model, default settings, ordered in the call.
        dict(name="point_scatter_1m", kind="point", mesh="knot", a=800, b=200, n=1000003, grid=0, lanes=0,
             dtype="f32"),
        # One step of fitting a million-triangle surface to a 256^3 distance grid: closest points and
        # the gradients of the points and vertices. The largest call.
        dict(name="point_train_256", kind="point_train", mesh="ico", a=223, b=0, n=256 ** 3, grid=256, lanes=64),
        # Rays that name their instance, many meshes in one launch (BatchedMesh), default tuning.
        dict(name="batch_4m", kind="batch", meshes=64, tri_max=50000, instances=64, n=1 << 22),
        # World rays through a scene of instances, the closest hit over all of them.
        dict(name="scene_ray_1m", kind="scene_ray", meshes=24, tri_max=50000, instances=512, n=1 << 20),
        # Closest point over the instances of a scene (collision, proximity).
        dict(name="scene_point_1m", kind="scene_point", meshes=24, tri_max=50000, instances=512, n=1 << 20),
        # A tree built from scratch on the device for a mesh whose topology changed.
        dict(name="build_1m", kind="build", mesh="ico", a=223, b=0),
    ]


def draw(rng):
    """One more case over the ranges that the listed ones stand for."""

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def mesh(most):
        if rng.random() < 0.5:
            tris = log_int(4000, most)
            b = max(8, int(math.sqrt(tris / 8)) + rng.randint(-3, 3))
            return dict(mesh="knot", a=max(16, tris // (2 * b)), b=b)
        return dict(mesh="ico", a=max(12, int(math.sqrt(log_int(4000, most) / 20)) - 1), b=0)

    kind = rng.choice(["ray", "ray", "ray_train", "ray_all", "point_host", "point", "point", "point_train", "batch",
                       "scene_ray", "scene_point", "build"])
    if kind == "ray":
        return dict(kind=kind, **mesh(1_000_000), n=log_int(200, 2_000_000), side=rng.choice(["front", "back", "double"]),
                    dtype=rng.choice(["f32", "f32", "f64"]))
    if kind == "ray_train":
        return dict(kind=kind, **mesh(1_000_000), n=log_int(4000, 1_500_000))
    if kind == "ray_all":
        return dict(kind=kind, **mesh(320_000), n=log_int(1000, 400_000), side=rng.choice(["front", "double"]))
    if kind == "point_host":
        return dict(kind=kind, **mesh(320_000), n=log_int(50, 200_000), dtype=rng.choice(["f32", "f64"]))
    if kind in ("point", "point_train"):
        grid = rng.choice([0, rng.randint(12, 160)])
        n = grid ** 3 if grid else log_int(1000, 2_000_000)
        lanes = rng.choice([0, 64]) if grid else 0
        if kind == "point_train":
            return dict(kind=kind, **mesh(1_000_000), n=n, grid=grid, lanes=lanes)
        return dict(kind=kind, **mesh(1_000_000), n=n, grid=grid, lanes=lanes, dtype=rng.choice(["f32", "f32", "f64"]))
    if kind == "batch":
        meshes = log_int(4, 64)
        return dict(kind=kind, meshes=meshes, tri_max=log_int(2000, 50000), instances=meshes * rng.randint(1, 3),
                    n=log_int(20_000, 4_000_000))
    if kind in ("scene_ray", "scene_point"):
        return dict(kind=kind, meshes=log_int(2, 24), tri_max=log_int(2000, 50000), instances=log_int(8, 700),
                    n=log_int(5000, 1_200_000))
    return dict(kind="build", **mesh(1_000_000))


# ---- what a program has in hand -------------------------------------------------------------------


@functools.lru_cache(maxsize=None)
def context(lanes):
    """One context and one stream per closest-point width, as a program keeps them."""
    ctx = M.Context(0)
    ctx.set_point_lanes(lanes)
    return ctx, torch.cuda.Stream()


@functools.lru_cache(maxsize=4)
def geometry(mesh, a, b):
    g = G.torus_knot(10, 3, a, b) if mesh == "knot" else G.displaced_icosphere(a)
    return g.ensure_index()


@functools.lru_cache(maxsize=4)
def geometries(count, tri_max):
    """Torus knots and spheres in turn, triangle counts log-uniform in [100, tri_max]."""
    rng = np.random.default_rng(count)
    out = []
    for i in range(count):
        t = float(np.exp(rng.uniform(np.log(100), np.log(tri_max))))
        if i % 2 == 0:
            radial = max(3, int(round(np.sqrt(t / 16))))
            out.append(G.torus_knot(rng.uniform(0.5, 2.0), rng.uniform(0.1, 0.5),
                                    max(3, int(round(t / (2 * radial)))), radial, 2, 3))
        else:
            rows = max(2, int(round(np.sqrt(t / 4))))
            out.append(G.sphere(rng.uniform(0.5, 2.0), max(3, int(round(t / (2 * rows)))), rows))
    return out


def upload(ctx, g):
    """The mesh in HBM with its SAH tree (leaves of 10), built on the device; the permuted index."""
    index = g.index.copy()
    tree = M.build(g.positions, index, strategy=M.SAH, target_leaf_size=10, ctx=ctx)
    return ctx.upload(tree, g.positions, index), index


def generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def unit(gen, n):
    v = torch.randn((n, 3), generator=gen, device="cuda", dtype=torch.float64)
    return v / v.norm(dim=1, keepdim=True)


def uniform(gen, lo, hi, n):
    lo, hi = (torch.as_tensor(x, dtype=torch.float64, device="cuda") for x in (lo, hi))
    return lo + (hi - lo) * torch.rand((n, 3), generator=gen, device="cuda", dtype=torch.float64)


def rays(gen, g, n):
    """Origins on a sphere around the model, each aimed at a uniform point of its box."""
    lo, hi = g.bounds()
    o = torch.as_tensor((lo + hi) / 2, device="cuda") + unit(gen, n) * (1.1 * float(np.linalg.norm(hi - lo)))
    d = uniform(gen, lo, hi, n) - o
    return o, d / d.norm(dim=1, keepdim=True)


def points(gen, g, n, grid):
    """The cell centres of a grid over the box enlarged by a tenth (shifted by up to half a cell, so
    that each seed has other points), or uniform points of that box."""
    lo, hi = g.bounds()
    mid, half = (lo + hi) / 2, (hi - lo) * 0.55
    lo, hi = mid - half, mid + half
    if not grid:
        return uniform(gen, lo, hi, n)
    step = torch.as_tensor((hi - lo) / grid, device="cuda")
    shift = torch.rand(3, generator=gen, device="cuda", dtype=torch.float64)
    axis = torch.arange(grid, device="cuda", dtype=torch.float64)
    z, y, x = torch.meshgrid(axis, axis, axis, indexing="ij")
    at = torch.stack([x, y, z], dim=-1).reshape(-1, 3)
    return torch.as_tensor(lo, device="cuda") + (at + shift) * step


def split(x):
    """float32 high and low parts of doubles."""
    hi = x.to(torch.float32)
    return hi, (x - hi.double()).to(torch.float32)


def hits(n):
    f = dict(dtype=torch.float32, device="cuda")
    return dict(face=torch.zeros(n, dtype=torch.int32, device="cuda"), distance=torch.zeros(n, **f),
                point=torch.zeros((n, 3), **f), barycoord=torch.zeros((n, 3), **f))


def instances(gen, geos, count):
    """A random geometry, rotation, scale (0.5 to 2) and place for each instance: column-major float32
    matrices, their inverses and the geometry of each."""
    q = torch.randn((count, 4), generator=gen, device="cuda", dtype=torch.float64)
    x, y, z, w = (q / q.norm(dim=1, keepdim=True)).unbind(1)
    r = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], dim=1).reshape(-1, 3, 3)
    scale = 0.5 + 1.5 * torch.rand((count, 1, 1), generator=gen, device="cuda", dtype=torch.float64)
    m = torch.zeros((count, 4, 4), device="cuda", dtype=torch.float64)
    m[:, :3, :3] = r * scale
    span = 6.0 * count ** (1 / 3)
    m[:, :3, 3] = (2 * torch.rand((count, 3), generator=gen, device="cuda", dtype=torch.float64) - 1) * span
    m[:, 3, 3] = 1
    world = m.transpose(1, 2).reshape(-1, 16).float().contiguous()
    inverse = torch.linalg.inv(world.double().reshape(-1, 4, 4)).reshape(-1, 16).float().contiguous()
    which = torch.randint(0, len(geos), (count,), generator=gen, device="cuda", dtype=torch.int32)
    return world, inverse, which


def world_boxes(geos, world, which):
    lo, hi = (torch.as_tensor(np.stack([g.bounds()[k] for g in geos]), device="cuda")[which.long()] for k in (0, 1))
    pick = torch.tensor([[(k >> j) & 1 for j in range(3)] for k in range(8)], device="cuda", dtype=torch.float64)
    corners = lo[:, None] + (hi - lo)[:, None] * pick[None]
    m = world.double().reshape(-1, 4, 4)  # row r is column r of the matrix
    at = corners @ m[:, :3, :3] + m[:, 3:, :3]
    return at.amin(dim=1), at.amax(dim=1)


def scene_setup(case, seed, ctx):
    gen = generator(seed)
    geos = geometries(case["meshes"], case["tri_max"])
    meshes, indices = [], []
    for g in geos:
        mesh, index = upload(ctx, g)
        meshes.append(mesh)
        indices.append(index)
    world, inverse, which = instances(gen, geos, case["instances"])
    lo, hi = world_boxes(geos, world, which)
    return gen, geos, meshes, indices, world, inverse, which, lo, hi


def prepare(case, seed):
    kind = case["kind"]
    ctx, stream = context(case.get("lanes", 0))
    s = dict(case=case, ctx=ctx, stream=stream, ptr=stream.cuda_stream)
    n = case.get("n", 0)
    if kind in ("batch", "scene_ray", "scene_point"):
        gen, geos, meshes, indices, world, inverse, which, lo, hi = scene_setup(case, seed, ctx)
        count = case["instances"]
        if kind == "batch":
            # rays split over the instances by a Zipf law over a random ranking, aimed at their boxes
            weight = 1.0 / torch.arange(1, count + 1, device="cuda", dtype=torch.float64) ** 1.1
            weight = weight[torch.randperm(count, generator=gen, device="cuda")]
            at = torch.multinomial(weight, n, replacement=True, generator=gen)
        else:
            at = torch.randint(0, count, (n,), generator=gen, device="cuda")
        target = lo[at] + (hi - lo)[at] * torch.rand((n, 3), generator=gen, device="cuda", dtype=torch.float64)
        s["out"] = hits(n)
        if kind == "scene_point":
            # points within a few units of random instances
            s["q"] = (target + 2.0 * torch.randn((n, 3), generator=gen, device="cuda", dtype=torch.float64)).float()
            s["order"] = torch.empty(n, dtype=torch.int32, device="cuda")
            s["work"] = torch.empty(M.Context.order_workspace_bytes(n), dtype=torch.uint8, device="cuda")
        else:
            if kind == "batch":
                r = (hi - lo)[at].norm(dim=1, keepdim=True)
                o = ((lo + hi)[at] / 2 + 1.5 * r * unit(gen, n)).float()
            else:
                a, b = lo.amin(dim=0), hi.amax(dim=0)
                o = ((a + b) / 2 + 0.625 * (b - a).norm() * unit(gen, n)).float()
            d = target - o.double()
            s["o"], s["d"] = o, (d / d.norm(dim=1, keepdim=True)).float()
        if kind == "batch":
            s["batch"] = ctx.batch(meshes)
            size = s["batch"].workspace_bytes(n)
            s.update(world=world, inverse=inverse, which=which, at=at.to(torch.int32).contiguous(),
                     work=torch.empty(size, dtype=torch.uint8, device="cuda"))
            p = {k: s[k].data_ptr() for k in ("world", "inverse")}
            p.update({k: v.data_ptr() for k, v in s["out"].items()})
            s["call"] = dict(p, instance_geometry=which.data_ptr(), n_instances=count, origins=s["o"].data_ptr(),
                             directions=s["d"].data_ptr(), ray_instance=s["at"].data_ptr(), n=n,
                             workspace=s["work"].data_ptr(), workspace_bytes=size)
        else:
            s["out"]["instance"] = torch.zeros(n, dtype=torch.int32, device="cuda")
            s["scene"] = ctx.scene(meshes, world.cpu().numpy(), inverse.cpu().numpy(),
                                   which.cpu().numpy().astype(np.uint32))
        torch.cuda.synchronize()
        return s

    g = geometry(case["mesh"], case["a"], case["b"])
    gen = generator(seed)
    if kind == "build":
        # the vertices of this seed: the model, slightly deformed
        phase = float(torch.rand(1, generator=gen, device="cuda"))
        p = torch.as_tensor(g.positions.reshape(-1, 3), device="cuda")
        s["positions"] = (p * (1.0 + 0.01 * torch.sin(7.0 * p[:, :1] + 6.28 * phase))).contiguous()
        s["index"] = torch.as_tensor(g.index.astype(np.uint32).view(np.int32), device="cuda")
        s["permuted"] = torch.zeros_like(s["index"])
        s["nodes"] = torch.zeros((2 * g.tri_count + 1) * 8, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        return s

    s["mesh"], s["mesh_index"] = upload(ctx, g)
    if kind == "point_host":
        q = points(gen, g, n, 0).cpu().numpy()
        s["q"] = q if case["dtype"] == "f64" else q.astype(np.float32)
        return s
    s["out"] = hits(n)
    if kind in ("ray", "ray_train", "ray_all"):
        o, d = rays(gen, g, n)
        s["side"] = dict(front=M.FRONT_SIDE, back=M.BACK_SIDE, double=M.DOUBLE_SIDE)[case.get("side", "front")]
        if case.get("dtype") == "f64":
            (s["o"], s["ol"]), (s["d"], s["dl"]) = split(o), split(d)
        else:
            s["o"], s["d"] = o.float(), d.float()
        if kind == "ray_all":
            s["room"] = 12 * n
            s["out"] = hits(s["room"])
            s["counts"] = torch.zeros(n, dtype=torch.int32, device="cuda")
            s["offsets"] = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    else:
        q = points(gen, g, n, case["grid"])
        if case.get("dtype") == "f64":
            s["q"], s["ql"] = split(q)
        else:
            s["q"] = q.float()
        s["order"] = torch.empty(n, dtype=torch.int32, device="cuda")
        s["work"] = torch.empty(M.Context.order_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    if kind in ("ray_train", "point_train"):
        f = dict(generator=gen, device="cuda", dtype=torch.float32)
        s["g_distance"] = torch.randn(n, **f)
        s["g_positions"] = torch.zeros((s["mesh"].vertex_count, 3), device="cuda")
        s["grad_work"] = torch.empty(M.Mesh.grad_workspace_bytes(n, M.GRAD_DETERMINISTIC), dtype=torch.uint8,
                                     device="cuda")
        if kind == "ray_train":
            s["g_barycoord"] = torch.randn((n, 3), **f)
            s["g_o"], s["g_d"] = torch.zeros((n, 3), device="cuda"), torch.zeros((n, 3), device="cuda")
            # the vertices after this step's update
            p = torch.as_tensor(g.positions.reshape(-1, 3), device="cuda")
            phase = 6.28 * float(torch.rand(1, generator=gen, device="cuda"))
            s["positions"] = (p * (1.0 + 0.01 * torch.sin(7.0 * p[:, :1] + phase))).contiguous()
        else:
            s["g_q"] = torch.zeros((n, 3), device="cuda")
    torch.cuda.synchronize()
    return s


# ---- one pass --------------------------------------------------------------------------------------


def run(s):
    return globals()["run_" + s["case"]["kind"]](s)


def out_ptrs(s):
    return [s["out"][k].data_ptr() for k in ("face", "distance", "point", "barycoord")]


def run_ray(s):
    n = s["case"]["n"]
    if s["case"]["dtype"] == "f64":
        s["mesh"].raycast_first_ff_d(s["o"].data_ptr(), s["ol"].data_ptr(), s["d"].data_ptr(), s["dl"].data_ptr(), n,
                                     *out_ptrs(s), side=s["side"], stream=s["ptr"])
    else:
        s["mesh"].raycast_first_d(s["o"].data_ptr(), s["d"].data_ptr(), n, *out_ptrs(s), side=s["side"],
                                  stream=s["ptr"])
    return s["out"]


def run_ray_train(s):
    n, m, out = s["case"]["n"], s["mesh"], s["out"]
    m.refit_d(s["positions"].data_ptr(), s["positions"].shape[0], stream=s["ptr"])
    m.raycast_first_d(s["o"].data_ptr(), s["d"].data_ptr(), n, *out_ptrs(s), side=s["side"], stream=s["ptr"])
    m.raycast_first_bwd_d(s["d"].data_ptr(), n, out["face"].data_ptr(), out["distance"].data_ptr(),
                          out["barycoord"].data_ptr(), s["g_distance"].data_ptr(), 0, s["g_barycoord"].data_ptr(),
                          s["g_o"].data_ptr(), s["g_d"].data_ptr(), s["g_positions"].data_ptr(), M.GRAD_DETERMINISTIC,
                          s["grad_work"].data_ptr(), s["grad_work"].numel(), stream=s["ptr"])
    return dict(out, g_o=s["g_o"], g_d=s["g_d"], g_positions=s["g_positions"])


def run_ray_all(s):
    n, m = s["case"]["n"], s["mesh"]
    m.raycast_count_d(s["o"].data_ptr(), s["d"].data_ptr(), n, s["counts"].data_ptr(), side=s["side"], stream=s["ptr"])
    with torch.cuda.stream(s["stream"]):
        torch.cumsum(s["counts"], 0, dtype=torch.int64, out=s["offsets"][1:])
    m.raycast_fill_d(s["o"].data_ptr(), s["d"].data_ptr(), n, s["offsets"].data_ptr(), s["room"], *out_ptrs(s),
                     side=s["side"], stream=s["ptr"])
    return dict(s["out"], offsets=s["offsets"])


def run_point_host(s):
    return s["mesh"].closest_point(s["q"])


def run_point(s):
    n = s["case"]["n"]
    s["ctx"].order_points_d(s["q"].data_ptr(), n, s["order"].data_ptr(), s["work"].data_ptr(), s["work"].numel(),
                            stream=s["ptr"])
    if "ql" in s:
        s["mesh"].closest_point_ff_d(s["q"].data_ptr(), s["ql"].data_ptr(), n, *out_ptrs(s), stream=s["ptr"],
                                     order_ptr=s["order"].data_ptr())
    else:
        s["mesh"].closest_point_d(s["q"].data_ptr(), n, *out_ptrs(s), stream=s["ptr"], order_ptr=s["order"].data_ptr())
    return s["out"]


def run_point_train(s):
    out = run_point(s)
    s["mesh"].closest_point_bwd_d(s["q"].data_ptr(), s["case"]["n"], out["face"].data_ptr(),
                                  out["distance"].data_ptr(), out["point"].data_ptr(), out["barycoord"].data_ptr(),
                                  s["g_distance"].data_ptr(), s["g_q"].data_ptr(), s["g_positions"].data_ptr(),
                                  M.GRAD_DETERMINISTIC, s["grad_work"].data_ptr(), s["grad_work"].numel(),
                                  stream=s["ptr"])
    return dict(out, g_q=s["g_q"], g_positions=s["g_positions"])


def run_batch(s):
    s["batch"].raycast_first_d(s["call"], stream=s["ptr"])
    return s["out"]


def run_scene_ray(s):
    out = s["out"]
    s["scene"].raycast_first_d(s["o"].data_ptr(), s["d"].data_ptr(), s["case"]["n"], out["face"].data_ptr(),
                               out["instance"].data_ptr(), out["distance"].data_ptr(), out["point"].data_ptr(),
                               out["barycoord"].data_ptr(), stream=s["ptr"])
    return out


def run_scene_point(s):
    n, out = s["case"]["n"], s["out"]
    s["ctx"].order_points_d(s["q"].data_ptr(), n, s["order"].data_ptr(), s["work"].data_ptr(), s["work"].numel(),
                            stream=s["ptr"])
    s["scene"].closest_point_d(s["q"].data_ptr(), n, out["face"].data_ptr(), out["instance"].data_ptr(),
                               out["distance"].data_ptr(), out["point"].data_ptr(), out["barycoord"].data_ptr(),
                               stream=s["ptr"], order_ptr=s["order"].data_ptr())
    return out


def run_build(s):
    # the build permutes the index it is given, so it gets a copy of the program's own
    with torch.cuda.stream(s["stream"]):
        s["permuted"].copy_(s["index"])
    tris = s["index"].numel() // 3
    count = s["ctx"].build_d(s["positions"].data_ptr(), s["positions"].shape[0], s["permuted"].data_ptr(), 4,
                             s["index"].numel(), [(0, tris)], s["nodes"].data_ptr(), s["nodes"].numel() * 4,
                             stream=s["ptr"])
    return dict(count=count[0], nodes=s["nodes"], index=s["permuted"])


# ---- what a pass cannot do without -------------------------------------------------------------------


def tri_count(case):
    if "mesh" in case:
        return 2 * case["a"] * case["b"] if case["mesh"] == "knot" else 20 * (case["a"] + 1) ** 2
    return case["meshes"] * (case["tri_max"] - 100) / math.log(case["tri_max"] / 100)


def work(case):
    """Queries and the mesh read once (three vertices and an index triplet per triangle, a quarter of a
    32-byte node), results written once; per query one walk down the tree (two boxes a level, 20
    operations each) and two triangles of 60 operations."""
    kind, tris = case["kind"], tri_count(case)
    if kind == "build":
        # vertices and index in, nodes and index out; per triangle and level a bin and a side
        return dict(bytes=tris * (36 + 12 + 12 + 9), flops=tris * 30 * math.log2(tris))
    n = case["n"]
    per_query = {"ray": 24 + 32, "ray_train": 24 + 32 + 16 + 24 + 32, "ray_all": 24 + 4 + 8 + 4 * 32, "point_host": 12 + 32,
                 "point": 12 + 32, "point_train": 12 + 32 + 4 + 12 + 32, "batch": 28 + 32, "scene_ray": 24 + 36,
                 "scene_point": 12 + 36}[kind]
    if case.get("dtype") == "f64":
        per_query += 24 if kind == "ray" else 12
    steps = math.log2(max(2.0, tris / max(1, case.get("meshes", 1)) / 10)) + math.log2(max(2, case.get("instances", 1)))
    return dict(bytes=n * per_query + tris * 56 + (72 * tris if kind in ("ray_train", "point_train") else 0),
                flops=n * (2 * 20 * steps + 2 * 60))


def tolerance(case):
    """Hits are decided exactly and their values rounded from about 48 bits, so two correct runs agree
    in the faces (ties in the last bits of the reference's own doubles aside) and to the last bits of
    float32 in the values; gradients are float32 sums of a few terms. Tree bytes are exact."""
    if case["kind"] == "build":
        return "exact"
    if case["kind"] in ("ray_train", "point_train"):
        return {"rel": 1e-5, "max": 1e-3, "differ": 1e-5}
    return {"rel": 1e-6, "max": 1e-3, "differ": 1e-5}


# ---- the same in 64 bits -----------------------------------------------------------------------------


def corners(positions, index):
    p = torch.as_tensor(np.asarray(positions).reshape(-1, 3).astype(np.float64), device="cuda")
    return [p[torch.as_tensor(index.astype(np.int64), device="cuda")[k::3]] for k in range(3)]


def blocks(n, tris, pairs=1 << 24):
    t = min(tris, 4096)
    q = max(1, min(n, pairs // t))
    for i in range(0, n, q):
        yield i, min(n, i + q), [(j, min(tris, j + t)) for j in range(0, tris, t)]


def first_hits(o, d, a, b, c, side):
    """The least ray parameter over all triangles and its triangle (-1 for none)."""
    n = o.shape[0]
    e1, e2 = b - a, c - a
    normal = torch.linalg.cross(e1, e2)
    best = torch.full((n,), INF, dtype=torch.float64, device="cuda")
    which = torch.full((n,), -1, dtype=torch.int64, device="cuda")
    for i, k, tiles in blocks(n, a.shape[0]):
        oo, dd = o[i:k], d[i:k]
        moment = torch.linalg.cross(dd, oo)
        for j, m in tiles:
            dn = dd @ normal[j:m].T
            # d . (Q x E2) with Q = o - a, and d . (E1 x Q)
            u = moment @ e2[j:m].T - dd @ torch.linalg.cross(a[j:m], e2[j:m]).T
            v = -(moment @ e1[j:m].T) - dd @ torch.linalg.cross(e1[j:m], a[j:m]).T
            qn = oo @ normal[j:m].T - (a[j:m] * normal[j:m]).sum(1)
            sign = torch.sign(dn)
            ok = (u * sign >= 0) & (v * sign >= 0) & ((u + v) * sign <= dn.abs()) & (qn * sign <= 0) & (dn != 0)
            if side != "double":
                ok &= (dn < 0) if side == "front" else (dn > 0)
            t = torch.where(ok, -qn / dn, INF)
            near, at = t.min(dim=1)
            better = near < best[i:k]
            best[i:k] = torch.where(better, near, best[i:k])
            which[i:k] = torch.where(better, at + j, which[i:k])
    return best, which


def hit_values(o, d, a, b, c, which):
    """Distance, point and barycoord of each hit, from its own triangle."""
    w = which.clamp(min=0)
    a, b, c = a[w], b[w], c[w]
    e1, e2, q = b - a, c - a, o - a
    det = (d * torch.linalg.cross(e1, e2)).sum(1)
    u = (d * torch.linalg.cross(q, e2)).sum(1) / det
    v = (d * torch.linalg.cross(e1, q)).sum(1) / det
    t = -(q * torch.linalg.cross(e1, e2)).sum(1) / det
    return t * d.norm(dim=1), o + t[:, None] * d, torch.stack([1 - u - v, u, v], dim=1)


def missed(which, *values):
    miss = which < 0
    return [torch.where(miss if v.dim() == 1 else miss[:, None], INF if v.dim() == 1 else float("nan"), v) for v in values]


def closest(q, a, b, c):
    """The least distance over all triangles and the point on the triangle that has it."""
    n = q.shape[0]
    best = torch.full((n,), INF, dtype=torch.float64, device="cuda")
    which = torch.zeros(n, dtype=torch.int64, device="cuda")
    for i, k, tiles in blocks(n, a.shape[0], 1 << 22):
        for j, m in tiles:
            _, d2 = closest_pairs(q[i:k, None], a[None, j:m], b[None, j:m], c[None, j:m])
            near, at = d2.min(dim=1)
            better = near < best[i:k]
            best[i:k] = torch.where(better, near, best[i:k])
            which[i:k] = torch.where(better, at + j, which[i:k])
    p, d2 = closest_pairs(q, a[which], b[which], c[which])
    return d2.sqrt(), p


def closest_pairs(q, a, b, c):
    def dot(x, y):
        return (x * y).sum(-1)

    e1, e2, r = b - a, c - a, q - a
    d11, d12, d22, r1, r2 = dot(e1, e1), dot(e1, e2), dot(e2, e2), dot(r, e1), dot(r, e2)
    det = d11 * d22 - d12 * d12
    v, w = (d22 * r1 - d12 * r2) / det, (d11 * r2 - d12 * r1) / det
    inside = (v >= 0) & (w >= 0) & (v + w <= 1)  # false for degenerate triangles (NaN)
    best = torch.where(inside[..., None], a + v[..., None] * e1 + w[..., None] * e2, a)
    least = torch.where(inside, dot(q - best, q - best), INF)
    for x, y in ((a, b), (a, c), (b, c)):
        e = y - x
        t = (dot(q - x, e) / dot(e, e)).nan_to_num(0.0).clamp(0, 1)
        p = x + t[..., None] * e
        d2 = dot(q - p, q - p)
        take = d2 < least
        best, least = torch.where(take[..., None], p, best), torch.where(take, d2, least)
    return best, least


def exact(case, seed):
    kind = case["kind"]
    if kind in ("build", "ray_all"):
        return None  # whole numbers; hits in the tree's own order
    if kind in ("batch", "scene_ray", "scene_point"):
        return exact_instances(case, seed)
    pairs = case["n"] * tri_count(case)
    if pairs > (PAIR_LIMIT // 3 if kind.startswith("point") else PAIR_LIMIT):
        return None
    s = prepare(case, seed)
    g = geometry(case["mesh"], case["a"], case["b"])
    if kind.startswith("point"):
        q = torch.as_tensor(s["q"], device="cuda").double()
        if "ql" in s:
            q = q + s["ql"].double()
        distance, p = closest(q, *corners(g.positions, g.index))
        out = dict(face=None, distance=distance, point=p, barycoord=None)
        if kind == "point_train":
            away = (q - p) / distance[:, None]
            out.update(g_q=away * s["g_distance"].double()[:, None], g_positions=None)
        return out
    o, d = s["o"].double(), s["d"].double()
    if "ol" in s:
        o, d = o + s["ol"].double(), d + s["dl"].double()
    positions = s["positions"].cpu().numpy() if kind == "ray_train" else g.positions
    a, b, c = corners(positions, g.index)
    _, which = first_hits(o, d, a, b, c, case.get("side", "front"))
    if kind == "ray":
        distance, p, bary = missed(which, *hit_values(o, d, a, b, c, which))
        return dict(face=None, distance=distance, point=p, barycoord=bary)
    p = torch.as_tensor(positions.astype(np.float64), device="cuda").requires_grad_()
    o.requires_grad_()
    d.requires_grad_()
    index = torch.as_tensor(g.index.astype(np.int64), device="cuda")
    distance, point, bary = hit_values(o, d, p[index[0::3]], p[index[1::3]], p[index[2::3]], which)
    hit = which >= 0
    loss = (distance * s["g_distance"])[hit].sum() + (bary * s["g_barycoord"])[hit].sum()
    g_o, g_d, g_p = torch.autograd.grad(loss, (o, d, p))
    distance, point, bary = missed(which, distance.detach(), point.detach(), bary.detach())
    return dict(face=None, distance=distance, point=point, barycoord=bary, g_o=g_o, g_d=g_d, g_positions=g_p)


def exact_instances(case, seed):
    n, kind = case["n"], case["kind"]
    s = prepare(case, seed)
    geos = geometries(case["meshes"], case["tri_max"])
    if kind == "batch":
        world, which = s["world"], s["which"]
    else:
        world, _, which = instances(generator(seed), geos, case["instances"])
    which = which.tolist()
    share = 1 if kind != "batch" else len(which)
    if n * sum(geos[k].tri_count for k in which) / share > PAIR_LIMIT // (3 if kind == "scene_point" else 1):
        return None
    best = torch.full((n,), INF, dtype=torch.float64, device="cuda")
    point = torch.full((n, 3), float("nan"), dtype=torch.float64, device="cuda")
    bary = point.clone()
    for k, which_k in enumerate(which):
        g, m = geos[which_k], world[k].double().reshape(4, 4)
        rows = (s["at"] == k).nonzero().reshape(-1) if kind == "batch" else torch.arange(n, device="cuda")
        if not rows.numel():
            continue
        a, b, c = (x @ m[:3, :3] + m[3, :3] for x in corners(g.positions, g.index))
        if kind == "scene_point":
            distance, p = closest(s["q"].double()[rows], a, b, c)
            w = p * float("nan")
        else:
            o, d = s["o"].double()[rows], s["d"].double()[rows]
            _, at = first_hits(o, d, a, b, c, "front")
            distance, p, w = missed(at, *hit_values(o, d, a, b, c, at))
        better = distance < best[rows]
        at = rows[better]
        best[at], point[at], bary[at] = distance[better], p[better], w[better]
    out = dict(face=None, distance=best, point=point, barycoord=None if kind == "scene_point" else bary)
    return out if kind == "batch" else dict(out, instance=None)
