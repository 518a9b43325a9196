"""A launch key off its default names the strategy's own kernel (seen by its
timing records: it writes partial rows that a second kernel adds, where the
kernel taken otherwise adds by itself at these sizes); the results are the
same."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev

pytestmark = pytest.mark.gpu

N, D, K = 1003, 7, 12
KEYS = [dict(vector_length=1), dict(vector_length=2), dict(global_size=4096), dict(local_size=64)]


def config(ctx, stage, strategy, keys):
    cfg = ctx.config(stage, strategy)
    for key, v in keys.items():
        if key in ("global_size", "local_size"):
            getattr(cfg, key)[0] = v
        else:
            setattr(cfg, key, v)
    return cfg


def records(ctx, fn):
    ctx.clear_records()
    ctx.profiling(True)
    fn()
    hip.synchronize()
    ctx.profiling(False)
    names = [name for name, _, _ in ctx.records()]
    ctx.clear_records()
    return [name for name in names if name != "SumGrid"]


@pytest.mark.parametrize("keys", [{}, dict(vector_length=4), dict(vector_length=8), dict(local_size=256)] + KEYS, ids=str)
@pytest.mark.parametrize("strategy", ["part_global", "part_local", "part_private"])
def test_mass_update(gpu_ctx, strategy, keys):
    lab = np.random.default_rng(3).integers(0, K, N).astype(np.uint32)
    masses, dl = dev(np.zeros(K, np.uint32)), dev(lab)
    cfg = config(gpu_ctx, clkmeans.STAGE_MASS_UPDATE, strategy, keys)
    names = records(gpu_ctx, lambda: gpu_ctx.mass_update(cfg, N, K, dl, masses))
    assert ("ReduceVectorParcol" in names) == (keys in KEYS)
    np.testing.assert_array_equal(masses.to_host(), np.bincount(lab, minlength=K))


@pytest.mark.parametrize("strategy,keys", [(s, k) for s in ("cluster_merge", "feature_sum", "feature_sum_pardim") for k in [{}] + KEYS]
                         + [("feature_sum_pardim", dict(local_features=2)), ("feature_sum_pardim", dict(thread_features=3)),
                            ("feature_sum_pardim", dict(local_features=3, thread_features=2, vector_length=2)),
                            ("feature_sum_pardim", dict(local_features=7))], ids=str)
def test_centroid_update(gpu_ctx, strategy, keys):
    rng = np.random.default_rng(4)
    pts, lab = rng.standard_normal((D, N)).astype(np.float32), rng.integers(0, K, N).astype(np.uint32)
    sums, dp, dl = dev(np.zeros((D, K))), dev(pts), dev(lab)
    cfg = config(gpu_ctx, clkmeans.STAGE_CENTROID_UPDATE, strategy, keys)
    names = records(gpu_ctx, lambda: gpu_ctx.centroid_update(cfg, D, N, K, dp, sums, dl))
    assert ("ReduceVectorParcol" in names) == bool(keys)
    if strategy == "feature_sum_pardim" and keys:
        assert "CentroidUpdateFeatureSumPardim" in names
    np.testing.assert_array_equal(sums.to_host(), O.sums_grid(pts, lab, K, O.grid_scales(pts)))
