"""The MFMA labeling's refinement takes a queue of a few thousand points about
as fast as one of 64: a work-group per 64 points, all of them at once."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev, zeros

pytestmark = pytest.mark.gpu


def refinement(ctx, n, d, k):
    rng = np.random.default_rng(n)
    pts = rng.standard_normal((d, n)).astype(np.float32)
    cen = np.ascontiguousarray(pts[:, :k])
    cen[:, k // 2:] = cen[:, :k // 2]  # every point between two equal ones: queued
    dp, dc, dl = dev(pts), dev(cen), zeros(n, np.uint32)
    cfg = ctx.config(clkmeans.STAGE_LABELING, "mfma_fp16")
    ctx.labeling(cfg, d, n, k, dp, dc, dl)
    hip.synchronize()
    np.testing.assert_array_equal(dl.to_host(), O.label(pts, cen))
    ctx.clear_records()
    ctx.profiling(True)
    for _ in range(10):
        ctx.labeling(cfg, d, n, k, dp, dc, dl)
    hip.synchronize()
    ctx.profiling(False)
    times = [ms for name, _, ms in ctx.records() if name == "LabelingMfmaRefine"]
    ctx.clear_records()
    assert len(times) == 10
    return min(times)


@pytest.mark.parametrize("d,k", [(24, 16), (100, 32)])
def test_queue_of_many_batches(gpu_ctx, d, k):
    one, many = refinement(gpu_ctx, 64, d, k), refinement(gpu_ctx, 8000, d, k)
    assert many <= 2.0 * one, (one, many)  # 1.2 measured; four batches to a work-group 2.9
