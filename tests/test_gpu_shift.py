"""The whole iteration's shift, for both types of points: it equals the largest
move of a non-empty cluster, recomputed in FP64 from the returned centroids,
whatever the output held before.  Once no label changes it is exactly zero for
float points (exact sums); double sums round in an order that is not fixed,
and leave it within what that rounding can move a centroid."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev, zeros

pytestmark = pytest.mark.gpu

# n, d, k on both sides of the lines between the passes: one and several
# clusters to a merge work-group, last groups that are not full, one value row
# per cluster and 65
F32 = [(1, 3, 1), (3000, 3, 5), (70001, 7, 33), (9001, 24, 48), (30011, 2, 150), (5000, 64, 37), (4100, 40, 300)]
F64 = [(1, 3, 1), (3000, 3, 5), (777, 1, 9), (30000, 5, 12), (20000, 8, 40), (200003, 4, 30), (150001, 12, 19), (1000003, 2, 33),
       (1000001, 4, 10), (9001, 24, 48), (60007, 32, 64), (50021, 32, 128), (4000, 32, 150), (2500, 16, 300)]


class Run:
    def __init__(self, ctx, pts, cen, strategy="cluster_merge"):
        f64 = pts.dtype == np.float64
        self.ctx, self.cfg = ctx, ctx.config(clkmeans.STAGE_FUSED, strategy)
        self.d, self.n = pts.shape
        self.k = cen.shape[1]
        self.pts, self.cen = dev(pts), [dev(cen), zeros(cen.shape, cen.dtype)]
        self.sums = zeros(cen.shape, np.float64)
        self.labels, self.masses = zeros(self.n, np.uint64 if f64 else np.uint32), zeros(self.k, np.uint64 if f64 else np.uint32)
        self.shift = dev(np.array([1e30]))  # what a caller left there

    def step(self):
        old, new = self.cen
        self.ctx.lloyd_step(self.cfg, self.d, self.n, self.k, self.pts, old, new, self.sums, self.labels, self.masses,
                            max_shift=self.shift)
        hip.synchronize()
        self.cen = [new, old]
        return float(self.shift.to_host()[0])


def data(n, d, k, dtype, spread=10.0):
    rng = np.random.default_rng(n + d + k)
    centres = rng.uniform(-spread, spread, (d, k))
    pts = (centres[:, np.arange(n) % k] + rng.standard_normal((d, n)) * 0.5).astype(dtype)
    cen = np.ascontiguousarray(pts[:, np.arange(k) % n])
    return pts, cen


@pytest.mark.parametrize("dtype,shape", [(np.float32, s) for s in F32] + [(np.float64, s) for s in F64],
                         ids=lambda v: "n%d_d%d_k%d" % v if isinstance(v, tuple) else v.__name__)
def test_shift_is_the_largest_move(gpu_ctx, dtype, shape):
    n, d, k = shape
    pts, cen = data(n, d, k, dtype)
    if k > 2:
        cen[:, k - 2] = 1e4  # stays empty
    r = Run(gpu_ctx, pts, cen)
    label = O.label_f64 if dtype == np.float64 else O.label
    for _ in range(3):
        old = r.cen[0].to_host()
        got = r.step()
        new, masses = r.cen[0].to_host(), r.masses.to_host()
        lab = label(pts, old)
        np.testing.assert_array_equal(r.labels.to_host(), lab)
        np.testing.assert_array_equal(masses, np.bincount(lab.astype(np.int64), minlength=k).astype(masses.dtype))
        move = np.sqrt(((new.astype(np.float64) - old.astype(np.float64)) ** 2).sum(0))[masses > 0]
        # the sum and the root in another order: d + 1 roundings of 2^-53
        assert abs(got - np.fmax.reduce(move)) <= 1e-12 * np.fmax.reduce(move)


@pytest.mark.parametrize("strategy", ["cluster_merge", "feature_sum"])
@pytest.mark.parametrize("dtype,shape", [(np.float32, s) for s in F32] + [(np.float64, s) for s in F64],
                         ids=lambda v: "n%d_d%d_k%d" % v if isinstance(v, tuple) else v.__name__)
def test_settled_shift(gpu_ctx, dtype, shape, strategy):
    n, d, k = shape
    pts, cen = data(n, d, k, dtype, spread=200.0)
    r = Run(gpu_ctx, pts, cen, strategy)
    settled, labels = 0, None
    for _ in range(300):
        old = r.cen[0].to_host()
        got = r.step()
        new, masses, before, labels = r.cen[0].to_host(), r.masses.to_host(), labels, r.labels.to_host()
        move = np.sqrt(((new.astype(np.float64) - old.astype(np.float64)) ** 2).sum(0))[masses > 0]
        assert abs(got - np.fmax.reduce(move)) <= 1e-12 * np.fmax.reduce(move)
        if settled and before is not None:  # this iteration and the last added the same points to every cell
            if dtype == np.float32:
                assert got == 0.0  # exact sums
            else:
                # two sums of m values in any order, m - 1 roundings of 2^-53
                # relative to the sum of |x| each, and a division each
                m = masses.astype(np.float64)
                absx = np.stack([np.bincount(labels.astype(np.int64), weights=np.abs(x), minlength=k) for x in pts])
                with np.errstate(all="ignore"):
                    off = 2 * (m * 2.0 ** -53 * absx / m + 2.0 ** -53 * np.abs(new))
                assert got <= np.fmax.reduce(np.sqrt((off ** 2).sum(0))[masses > 0])
        settled = settled + 1 if before is not None and np.array_equal(labels, before) else 0
        if settled == 4:
            break
    assert settled == 4
