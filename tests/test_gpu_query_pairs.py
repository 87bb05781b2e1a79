"""Distance-map queries of many points (two threads a point) against the same
points in calls of fewer (one thread a point, held to the oracle elsewhere),
bit for bit: points inside, outside, on the box's faces and not finite, with
and without the optional outputs."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1 << 17, (1 << 17) + 1, 200003])
@pytest.mark.parametrize("cells", [(7, 5, 9), (40, 33, 21)])
def test_many_points_equal_few(gpu_ctx, n, cells):
    from fullc0ntact_amd import _lib, meshes
    from fullc0ntact_amd.distance_map import DistanceMap
    print(n, cells, flush=True)
    v, f = meshes.torus_knot(2, 3, 64, 8, radius=0.12, scale=0.25, center=(0.0, 0.0, 0.0))
    m = DistanceMap.from_mesh(gpu_ctx, v, f, cells, 2.0 / max(cells), (-1.0, -1.0, -1.0))
    rng = np.random.default_rng(n)
    lo, hi = np.float32(m.bmin), np.float32(m.bmax)
    q = rng.uniform(lo - 0.1, hi + 0.1, (n, 3)).astype(np.float32)
    q[::97, 0] = hi[0]
    q[1::97, 1] = lo[1]
    q[2::97] = hi
    q[3::997, 2] = np.nan
    q[4::997, 1] = np.inf
    d, c, w = m.query(q)
    parts = [m.query(q[i:i + 50000]) for i in range(0, n, 50000)]
    for k, whole in enumerate((d, c, w)):
        few = np.concatenate([p[k] for p in parts])
        assert np.array_equal(whole.view(np.uint32), few.view(np.uint32)), k
    assert np.any(d == 5.0) and np.any(d < 0.3)
    # no closest points, no normals
    dp = _lib.DeviceArray.from_host(gpu_ctx, q)
    dd = _lib.DeviceArray(gpu_ctx, 4 * n)
    _lib.check(_lib.lib.fc_distmap_query(gpu_ctx.handle, m.handle, dp.ptr, n, dd.ptr, None, None))
    gpu_ctx.sync()
    assert np.array_equal(dd.download(np.float32, n).view(np.uint32), d.view(np.uint32))
