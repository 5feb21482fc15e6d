"""The refit's run of small depths in one workgroup, at its edges: one node, trees of few depths, depths
of about 1,024 nodes, more depths than a run holds, several roots. The nodes are the oracle's."""
import numpy as np
import pytest

import mbvh_amd as M
from mbvh_amd import geometry as G
import oracle_py as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = M.Context(0)
    yield c
    c.close()


def check(ctx, positions, index, **opts):
    index = np.ascontiguousarray(index, dtype=np.uint32)
    tree = M.build(positions, index, **opts)
    mesh = ctx.upload(tree, positions, index)
    rng = np.random.default_rng(1)
    for scale in (0.2, 0.0):
        pos = (positions.reshape(-1, 3) * (1 + scale * rng.normal(size=(positions.size // 3, 3)))).astype(np.float32)
        om = O.OracleMesh(pos, index, tree.roots, indirect=tree.indirect)
        for a, b in zip(mesh.refit(pos), om.refit()):
            np.testing.assert_array_equal(a, b)
    mesh.free()


@pytest.mark.parametrize("triangles", [1, 2, 3, 1023, 1024, 1025, 2047, 2049, 4100])
def test_depths(ctx, triangles):
    p = np.random.default_rng(triangles).uniform(-1, 1, size=(3 * triangles, 3)).astype(np.float32)
    check(ctx, p, np.arange(3 * triangles), target_leaf_size=1)


@pytest.mark.parametrize("triangles", [47, 48, 49, 100])
def test_more_depths_than_a_run(ctx, triangles):
    """Triangles at powers of two: each split at the centre parts off one of them."""
    at = 2.0 ** np.arange(triangles)[:, None, None]
    p = (at * np.array([[1, 0, 0], [1.1, 0, 0], [1, 0.1, 0]])[None]).reshape(-1, 3).astype(np.float32)
    check(ctx, p, np.arange(3 * triangles), strategy=M.CENTER, target_leaf_size=1, max_depth=150)
