"""The centroid update's slices for few points, where they get narrower so that
enough work-groups run: grid-exact sums at the edges of that rule, and no great
difference between random labels and every point in one cluster."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev
from tests.test_gpu_split_fallback import micros

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,k", [(511, 128, 30), (512, 128, 30), (1199, 64, 300), (1200, 64, 300), (4097, 16, 64), (8191, 20, 1500),
                                   (9601, 33, 130), (33000, 3, 500), (70001, 100, 40), (70001, 5, 2000)])
@pytest.mark.parametrize("same", [False, True])
def test_sums(gpu_ctx, n, d, k, same):
    rng = np.random.default_rng(n + d + k)
    pts = (rng.standard_normal((d, n)) * 3).astype(np.float32)
    lab = (np.full(n, k - 1) if same else rng.integers(0, k, n)).astype(np.uint32)
    sums = dev(np.zeros((d, k)))
    gpu_ctx.centroid_update(gpu_ctx.config(clkmeans.STAGE_CENTROID_UPDATE, "feature_sum"), d, n, k, dev(pts), sums, dev(lab))
    hip.synchronize()
    np.testing.assert_array_equal(sums.to_host(), O.sums_grid(pts, lab, k, O.grid_scales(pts)))


# One cluster takes all of a wave's additions to a few cells: 1.2 to 1.5 times
# the time of random labels with the narrower slices, 2.6 to 3.1 in a few wide
# ones.
@pytest.mark.parametrize("n,d,k", [(3000, 8, 300), (3000, 20, 700), (8000, 20, 1500)])
def test_time(gpu_ctx, n, d, k):
    rng = np.random.default_rng(1)
    dp, sums = dev(rng.standard_normal((d, n)).astype(np.float32)), dev(np.zeros((d, k)))
    spread, same = dev(rng.integers(0, k, n).astype(np.uint32)), dev(np.zeros(n, np.uint32))
    cfg = gpu_ctx.config(clkmeans.STAGE_CENTROID_UPDATE, "feature_sum")
    gpu_ctx.sum_grid_from_points(d, n, dp)
    try:
        t = [micros(lambda: gpu_ctx.centroid_update(cfg, d, n, k, dp, sums, lab)) for lab in (same, spread)]
    finally:
        gpu_ctx.sum_grid_clear()
    assert t[0] <= 1.9 * t[1], t
