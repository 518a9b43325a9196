"""The strategies' own kernels where the sizes would otherwise take another one:
the private-column and the bounded fused pass, four points per work-item in
work-groups of 256, and the three centroid-update kernels, under a geometry
that names them; and the first sizes above the line from where the fused ones
are taken by themselves.  Odd numbers of points, buffers that start 4 bytes off,
ties and duplicated centroids.  Labels, masses and grid sums equal the oracle's."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev, zeros

pytestmark = pytest.mark.gpu


def data(n, d, k, kind):
    rng = np.random.default_rng(n + 31 * d + k)
    if kind == "lattice":
        pts = rng.integers(-2, 3, (d, n)).astype(np.float32)
    else:
        pts = (rng.uniform(-9, 9, (d, k))[:, rng.integers(0, k, n)] + rng.standard_normal((d, n))).astype(np.float32)
    cen = np.ascontiguousarray(pts[:, np.arange(k) % n])
    if k > 3:
        cen[:, 3] = cen[:, 1]
    return pts, cen, rng


def run_fused(ctx, pts, cen, start, strategy, **keys):
    d, n = pts.shape
    k = cen.shape[1]
    dp = dev(np.concatenate([np.zeros(1, np.float32), pts.reshape(-1)]))
    dl = dev(np.concatenate([np.full(1, 0xDEAD, np.uint32), start]))
    sums, masses = dev(np.zeros((d, k))), dev(np.zeros(k, np.uint32))
    cfg = ctx.config(clkmeans.STAGE_FUSED, strategy)
    for key, v in keys.items():
        getattr(cfg, key)[0] = v
    ctx.clear_records()
    ctx.profiling(True)
    ctx.fused(cfg, d, n, k, dp.offset(1), dev(cen), sums, dl.offset(1), masses)
    hip.synchronize()
    ctx.profiling(False)
    names = [name for name, _, _ in ctx.records()]
    ctx.clear_records()
    lab = dl.to_host()
    assert lab[0] == 0xDEAD
    return names, lab[1:], masses.to_host(), sums.to_host()


def check(ctx, n, d, k, kind, strategy, name, **keys):
    pts, cen, rng = data(n, d, k, kind)
    scales = O.grid_scales(pts)
    starts = [rng.integers(0, 2 ** 32, n, dtype=np.uint64).astype(np.uint32)]
    for turn in range(3):
        ref = O.label(pts, cen)
        for start in starts:
            names, lab, masses, sums = run_fused(ctx, pts, cen, start, strategy, **keys)
            assert name in names
            np.testing.assert_array_equal(lab, ref)
            np.testing.assert_array_equal(masses, np.bincount(ref, minlength=k))
            np.testing.assert_array_equal(sums, O.sums_grid(pts, ref, k, scales))
        starts = [ref]  # the labels of the iteration before
        with np.errstate(all="ignore"):
            cen = (sums / masses.astype(np.float64)).astype(np.float32)


@pytest.mark.parametrize("strategy,name", [("cluster_merge", "FusedClusterMerge"), ("cluster_merge_bounded", "FusedClusterMergeBounded")])
@pytest.mark.parametrize("kind", ["blobs", "lattice"])
@pytest.mark.parametrize("n,d,k", [(3, 4, 2), (30001, 1, 7), (30002, 2, 10), (30003, 3, 9), (65537, 4, 10), (20005, 4, 24), (9999, 5, 9),
                                   (4097, 8, 8), (4098, 8, 12), (3001, 16, 6), (3002, 32, 3)])
def test_named(gpu_ctx, n, d, k, kind, strategy, name):
    check(gpu_ctx, n, d, k, kind, strategy, name, global_size=256 * 61)


@pytest.mark.parametrize("strategy,name", [("cluster_merge", "FusedClusterMerge"), ("cluster_merge_bounded", "FusedClusterMergeBounded")])
@pytest.mark.parametrize("kind", ["blobs", "lattice"])
@pytest.mark.parametrize("extra,d,k", [(3, 4, 10), (1, 2, 10), (2, 3, 5)])
def test_from_four_million_points(gpu_ctx, extra, d, k, kind, strategy, name):
    check(gpu_ctx, (4 << 20) + extra, d, k, kind, strategy, name)


@pytest.mark.parametrize("strategy,name", [("cluster_merge", "CentroidUpdateClusterMerge"), ("feature_sum", "CentroidUpdateFeatureSum"),
                                           ("feature_sum_pardim", "CentroidUpdateFeatureSumPardim")])
@pytest.mark.parametrize("n,d,k", [(5, 1, 2), (30001, 4, 10), (30003, 7, 9), (20002, 16, 5), (4099, 30, 2), (70001, 3, 16)])
def test_centroid_update(gpu_ctx, n, d, k, strategy, name):
    pts, _, rng = data(n, d, k, "blobs")
    pts[0, n // 2], pts[d - 1, n // 3] = np.nan, np.inf
    lab = rng.integers(0, k, n).astype(np.uint32)
    dp = dev(np.concatenate([np.zeros(1, np.float32), pts.reshape(-1)]))
    dl = dev(np.concatenate([np.zeros(1, np.uint32), lab]))
    ref = O.sums_grid(pts, lab, k, O.grid_scales(pts))
    for keys in (dict(global_size=256 * 61), dict(local_features=4, thread_features=1), dict(local_features=2, thread_features=3)):
        if strategy != "feature_sum_pardim" and "global_size" not in keys:
            continue
        cfg = gpu_ctx.config(clkmeans.STAGE_CENTROID_UPDATE, strategy)
        for key, v in keys.items():
            if key == "global_size":
                cfg.global_size[0] = v
            else:
                setattr(cfg, key, v)
        sums = zeros((d, k), np.float64)
        gpu_ctx.clear_records()
        gpu_ctx.profiling(True)
        gpu_ctx.centroid_update(cfg, d, n, k, dp.offset(1), sums, dl.offset(1))
        hip.synchronize()
        gpu_ctx.profiling(False)
        names = [x for x, _, _ in gpu_ctx.records()]
        gpu_ctx.clear_records()
        assert name in names and "ReduceVectorParcol" in names
        np.testing.assert_array_equal(sums.to_host(), ref)
