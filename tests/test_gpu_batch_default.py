"""The batched launch's own choice of lanes (no tuning given, none measured) on both sides of its line:
the results of the shapes it chooses between."""
import numpy as np
import pytest

import mbvh_amd as M
from test_gpu_batch import _host, _outputs, _params, case, ctx, torch  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 30000])
def test_default_shape(case, n):  # noqa: F811
    w, _, meshes, _, D, wsb = case
    fresh = meshes[0].ctx.batch(meshes)
    results = []
    for t in (None, M.BatchTuning(4, 16, 64, 4, 0.0), M.BatchTuning(1, 8, 64, 4, 0.0)):
        out = _outputs(n)
        fresh.raycast_first_d(_params(w, D, out, wsb, n), tuning=t)
        torch.cuda.synchronize()
        results.append(_host(out))
    fresh.free()
    for r in results[1:]:
        for k in r:
            np.testing.assert_array_equal(r[k].view(np.uint32), results[0][k].view(np.uint32), err_msg=k)
