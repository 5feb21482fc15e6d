"""The bounds of the triangle frames (csrc/mbvh_frame.h) against exact rational distances, on the host:
the header compiled with contraction on, as for the device. A frame's d2 - e2 is a lower bound of the
triangle's squared distance, d2 + e2 an upper one, also for triangles that are segments or nearly."""
import ctypes
import os
import shutil
import subprocess
from fractions import Fraction as F

import numpy as np
import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "frame_host")


@pytest.fixture(scope="module")
def frames(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    so = str(tmp_path_factory.mktemp("frame") / "frame_host.so")
    fma = ["-mfma"] if os.path.exists("/proc/cpuinfo") and " fma " in open("/proc/cpuinfo").read() else []
    subprocess.run([cxx, "-std=c++17", "-O2", *fma, "-ffp-contract=fast", "-w", "-shared", "-fPIC", "-I" + HERE,
                    os.path.join(HERE, "frame_host.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)

    def run(tris, queries):
        tris = np.ascontiguousarray(tris, np.float32)
        queries = np.ascontiguousarray(queries, np.float32)
        out = np.zeros((len(tris), 3), np.float32)
        p = ctypes.c_void_p
        lib.frame_distances(p(tris.ctypes.data), p(queries.ctypes.data), len(tris), p(out.ctypes.data))
        return out

    return run


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _sub(a, b):
    return [a[0] - b[0], a[1] - b[1], a[2] - b[2]]


def _cross(a, b):
    return [a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]


def exact_dist2(tri, q):
    """The exact squared distance from q to the triangle (rational arithmetic)."""
    a, b, c = ([F(float(x)) for x in v] for v in tri)
    q = [F(float(x)) for x in q]
    best = None
    for s, e in ((a, b), (b, c), (c, a)):
        d, r = _sub(e, s), _sub(q, s)
        ll = _dot(d, d)
        t = min(max(_dot(r, d) / ll, F(0)), F(1)) if ll else F(0)
        v = [r[k] - t * d[k] for k in range(3)]
        best = _dot(v, v) if best is None else min(best, _dot(v, v))
    n = _cross(_sub(b, a), _sub(c, a))
    nn = _dot(n, n)
    if nn and all(_dot(_cross(_sub(e, s), _sub(q, s)), n) >= 0 for s, e in ((a, b), (b, c), (c, a))):
        best = min(best, _dot(_sub(q, a), n) ** 2 / nn)
    return best


def _tris(kind, rng, n):
    if kind.startswith("line"):  # exactly collinear, distinct corners, in any order: a + i e with whole i
        step = 1.0 / int(kind[4:])
        e = rng.integers(-40, 41, (n, 1, 3)) * step
        e[np.abs(e).sum((1, 2)) == 0] = step
        i = np.stack([rng.permutation(7)[:3] - 3 for _ in range(n)])[:, :, None]
        return rng.integers(-200, 201, (n, 1, 3)) * step + i * e
    a, b, c = rng.standard_normal((3, n, 3)).astype(np.float32)
    if kind == "equal":
        k = np.arange(n) % 4
        return np.stack([a, np.where((k == 0)[:, None] | (k == 3)[:, None], a, b),
                         np.where((k == 1)[:, None], b, np.where((k == 2)[:, None] | (k == 3)[:, None], a, c))], 1)
    # an apex off the middle of a b, or off a = 0 (where floats resolve it), by 2^-k of its length
    h = 2.0 ** -rng.integers(8, 50, (n, 1))
    a[::2] = 0
    mid = np.where((np.arange(n) % 2 == 0)[:, None], 0, rng.uniform(0.1, 0.9, (n, 1)))
    t = np.stack([a, b, a + (b - a) * mid + c * h], 1)
    return np.stack([x[rng.permutation(3)] for x in t])


@pytest.mark.parametrize("kind", ["line1", "line256", "line65536", "equal", "thin"])
@pytest.mark.parametrize("far", [0.02, 0.5, 30.0])
def test_bounds_hold(frames, kind, far):
    rng = np.random.default_rng(41)
    tris = np.asarray(_tris(kind, rng, 500)).astype(np.float32)
    size = np.abs(tris.max(1) - tris.min(1)).max(1)[:, None]
    w = rng.dirichlet([1, 1, 1], len(tris))
    q = ((w[:, :, None] * tris).sum(1) + far * size * rng.standard_normal((len(tris), 3))).astype(np.float32)
    out = frames(tris, q)
    same_ab = (tris[:, 0] == tris[:, 1]).all(1) & ~(tris[:, 1] == tris[:, 2]).all(1)
    for t, p, (d2, e2, wide), ab in zip(tris, q, out, same_ab):
        exact = exact_dist2(t, p)
        assert F(float(d2)) - F(float(e2)) <= exact, (t, p, d2, e2, float(exact))
        assert exact <= F(float(d2)) + F(float(e2)), (t, p, d2, e2, float(exact))
    if kind == "equal":  # segments bound the search, except a, a, b, whose exact closest point can be NaN
        assert np.array_equal(np.signbit(out[:, 2]), same_ab)
    if kind.startswith("line"):
        assert np.signbit(out[:, 2]).all()


@pytest.mark.parametrize("corner", [0, 1, 2])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_a_corner_that_is_not_finite(frames, corner, value):
    t = np.arange(9, dtype=np.float32).reshape(1, 3, 3) ** 2
    t[0, corner, 1] = value
    out = frames(t, np.zeros((1, 3), np.float32))
    assert np.isnan(out[0, 2]) and np.isnan(out[0, 0] - out[0, 1])
