"""The MFMA labeling's point queue and its refinement, with every point queued
(duplicate centroids tie exactly): tables with and without room for the waves'
queue entries in LDS, several 64-point steps a wave, fewer and more tiles of 16
centroids than the refinement's waves -- labels equal the oracle's.  Then the
division without a shift at the edges of its grid."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev, zeros

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d,k", [
    (70, 5, 1), (4000, 17, 2), (4000, 32, 16), (4000, 33, 17), (4000, 40, 48), (4000, 24, 65),
    (3000, 32, 136 * 16), (3000, 32, 136 * 16 + 1), (3000, 64, 72 * 16), (3000, 64, 72 * 16 + 3),
    (2000, 96, 50 * 16), (2000, 70, 51 * 16), (2000, 128, 38 * 16), (300 * 4099, 12, 40), (100 * 4099, 100, 30),
])
@pytest.mark.parametrize("strategy", ["mfma_bf16", "mfma_fp16"])
def test_all_points_queued(gpu_ctx, strategy, n, d, k):
    rng = np.random.default_rng(n + d + k)
    base = min(n, 4099)
    pts = rng.standard_normal((d, base)).astype(np.float32)
    cen = rng.standard_normal((d, k)).astype(np.float32)
    if k > 1:
        cen[:, (k + 1) // 2:] = cen[:, :k // 2]
    pts = np.ascontiguousarray(pts)
    ref = np.tile(O.label(pts, cen), n // base)
    pts = np.ascontiguousarray(np.tile(pts, (1, n // base)))
    dl = zeros(n, np.uint32)
    gpu_ctx.labeling(gpu_ctx.config(clkmeans.STAGE_LABELING, strategy), d, n, k, dev(pts), dev(cen), dl)
    hip.synchronize()
    np.testing.assert_array_equal(dl.to_host(), ref)


@pytest.mark.parametrize("d,k", [(1, 1), (3, 85), (4, 64), (1, 257), (64, 1024), (7, 1300)])
def test_divide_values(gpu_ctx, d, k):
    rng = np.random.default_rng(d * k)
    sums = rng.standard_normal((d, k)) * 1e3
    masses = rng.integers(0, 50, k).astype(np.uint32)
    masses[0] = 0  # an empty cluster: the quotient as it comes
    sums[0, 0] = 0.0
    cen, shift = zeros((d, k), np.float32), zeros(1, np.float64)
    with np.errstate(all="ignore"):
        ref = (sums / masses.astype(np.float64)).astype(np.float32)
    for kw in ({}, {"old_centroids": dev(np.ones((d, k), np.float32))}, {"max_shift": shift}):
        gpu_ctx.divide(d, k, dev(sums), dev(masses), cen, **kw)
        hip.synchronize()
        np.testing.assert_array_equal(cen.to_host().reshape(d, k), ref)
    assert shift.to_host()[0] == 0.0
