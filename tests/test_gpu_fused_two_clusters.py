"""Two clusters of many features: the fused pass takes the plain kernel, which
is the faster one, under an automatic geometry too."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev, zeros
from tests.test_gpu_split_fallback import micros

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d", [(400000, 32), (1000003, 20)])
def test_two_clusters(gpu_ctx, n, d):
    k = 2
    pts, _ = clkmeans.generate_blobs(n, d, k, sigma=1.0, box=10.0, seed=1)
    cen = np.ascontiguousarray(pts[:, :k])
    dp, dc, dl = dev(pts), dev(cen), zeros(n, np.uint32)
    new, sums, masses = zeros((d, k), np.float32), zeros((d, k), np.float64), zeros(k, np.uint32)
    auto, named = (gpu_ctx.config(clkmeans.STAGE_FUSED, "cluster_merge") for _ in range(2))
    named.global_size[0] = 256 * 512
    gpu_ctx.sum_grid_from_points(d, n, dp)
    try:
        t = [micros(lambda: gpu_ctx.lloyd_step(c, d, n, k, dp, dc, new, sums, dl, masses)) for c in (auto, named)]
        hip.synchronize()
        ref = O.label(pts, cen)
        gpu_ctx.lloyd_step(auto, d, n, k, dp, dc, new, sums, dl, masses)
        hip.synchronize()
    finally:
        gpu_ctx.sum_grid_clear()
    np.testing.assert_array_equal(dl.to_host(), ref)
    np.testing.assert_array_equal(masses.to_host(), np.bincount(ref, minlength=k))
    assert t[0] <= 1.15 * t[1], t  # 1.4 with split labels
