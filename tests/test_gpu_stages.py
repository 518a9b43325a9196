"""The mass histogram and the centroid-update cell kernel at the edges of
their sizes: exact counts and grid-exact sums against the oracle, added to
what the outputs held (one rounding), labels >= k skipped."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev

pytestmark = pytest.mark.gpu

MASS = ["global_atomic", "part_global", "part_local", "part_private"]


@pytest.mark.parametrize("k", [1, 7, 40, 513, 16384, 16385])
@pytest.mark.parametrize("n", [1, 3, 64, 4099, 262144, 700001])
def test_mass_histogram(gpu_ctx, n, k):
    rng = np.random.default_rng(n + k)
    lab = rng.integers(0, k + max(k // 8, 1), n).astype(np.uint32)  # some are not labels
    before = rng.integers(0, 1000, k).astype(np.uint32)
    ref = before + np.bincount(lab[lab < k], minlength=k).astype(np.uint32)
    padded = dev(np.concatenate([np.zeros(1, np.uint32), lab]))  # rows that start 4 bytes off
    for strategy in MASS:
        masses = dev(before)
        cfg = gpu_ctx.config(clkmeans.STAGE_MASS_UPDATE, strategy)
        gpu_ctx.mass_update(cfg, n, k, padded.offset(1), masses)
        hip.synchronize()
        np.testing.assert_array_equal(masses.to_host(), ref)


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("n,d,k", [
    (1, 1, 1), (63, 2, 3), (65, 3, 2), (1000, 5, 33), (4097, 9, 1), (5000, 16, 300), (5001, 17, 700), (6000, 70, 40),
    (30001, 4, 5000), (3000, 3, 17000), (3000, 2, 20000), (600003, 6, 10),
    # one work-group per slice adds to the sums itself, and one point more
    (16384, 1, 30), (16385, 2, 7), (8192, 3, 10), (8193, 4, 10), (4096, 7, 300), (4097, 8, 5), (2048, 33, 40), (2049, 64, 9),
])
def test_centroid_cells(gpu_ctx, n, d, k, special):
    rng = np.random.default_rng(n + d + k)
    pts = (rng.standard_normal((d, n)) * 5).astype(np.float32)
    if special:
        pts[0, n // 2], pts[d - 1, n // 3], pts[d // 2, n // 4] = np.nan, np.inf, -np.inf
    lab = rng.integers(0, k, n).astype(np.uint32)
    before = rng.standard_normal((d, k))
    ref = before + O.sums_grid(pts, lab, k, O.grid_scales(pts))
    dp, dl = dev(pts), dev(lab)
    for strategy in ("cluster_merge", "feature_sum", "feature_sum_pardim"):
        sums = dev(before)
        cfg = gpu_ctx.config(clkmeans.STAGE_CENTROID_UPDATE, strategy)
        gpu_ctx.centroid_update(cfg, d, n, k, dp, sums, dl)
        hip.synchronize()
        if k <= 17000:
            np.testing.assert_array_equal(sums.to_host(), ref)
        else:  # global atomics: rounded at every addition to what was there
            np.testing.assert_allclose(sums.to_host(), ref, rtol=1e-12, atol=1e-12)
