"""Split-operand MFMA labels (clk_split.hpp) at the edges of its shapes: the
labels, masses and grid-exact sums equal the oracle's, exactly."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev, zeros

pytestmark = pytest.mark.gpu

SHAPES = [  # n, d, k: operand forms of 8, 16, 32 .. 128 features, tile and batch remainders
    (5000, 1, 130), (4096, 2, 64), (4097, 3, 100), (70001, 7, 33), (6000, 8, 16), (5555, 8, 17), (4160, 9, 31),
    (30003, 13, 48), (5000, 16, 97), (4500, 17, 15), (9001, 24, 48), (4100, 32, 256), (6001, 33, 40), (4200, 64, 129),
    (4111, 65, 30), (4100, 96, 65), (4099, 97, 33), (4096, 128, 100), (5000, 5, 1200), (4300, 30, 700),
]


def points(n, d, k, kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "blobs":  # overlapping: many undecided points
        return clkmeans.generate_blobs(n, d, k, sigma=2.0, box=8.0, seed=seed)[0]
    if kind == "lattice":  # exact ties and duplicated centroids
        return rng.integers(-3, 4, (d, n)).astype(np.float32)
    if kind == "offset":  # large norms against small gaps
        return (rng.standard_normal((d, n)) + 300.0).astype(np.float32)
    p = rng.standard_normal((d, n)).astype(np.float32)  # "special"
    p *= np.float32(2.0) ** rng.integers(-130, 100, n).astype(np.float32)
    p[0, 7::53], p[d - 1, 9::59], p[0, 11::61] = np.nan, np.inf, -np.inf
    return p


def centroids(pts, k, kind):
    c = np.ascontiguousarray(pts[:, np.arange(k) * 2 % pts.shape[1]])
    if kind == "special":
        c[~np.isfinite(c)] = 1.0
        c[0, k // 2] = np.nan
        c[0, k // 3] = np.inf
    return c


@pytest.mark.parametrize("kind", ["blobs", "lattice", "offset", "special"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "n%d_d%d_k%d" % s)
def test_split_labels_and_sums(gpu_ctx, shape, kind):
    n, d, k = shape
    pts = points(n, d, k, kind, n + d + k)
    cen = centroids(pts, k, kind)
    ref = O.label(pts, cen)
    dp, dc = dev(pts), dev(cen)
    labels = dev(np.full(n, 0xFFFFFFFF, np.uint32))
    gpu_ctx.labeling(gpu_ctx.config(clkmeans.STAGE_LABELING, "unroll_vector"), d, n, k, dp, dc, labels)
    hip.synchronize()
    np.testing.assert_array_equal(labels.to_host(), ref)
    labels = dev(np.full(n, 0xFFFFFFFF, np.uint32))
    sums, masses = zeros((d, k), np.float64), zeros(k, np.uint32)
    gpu_ctx.fused(gpu_ctx.config(clkmeans.STAGE_FUSED, "feature_sum"), d, n, k, dp, dc, sums, labels, masses)
    hip.synchronize()
    np.testing.assert_array_equal(labels.to_host(), ref)
    np.testing.assert_array_equal(masses.to_host(), O.mass(ref, k))
    np.testing.assert_array_equal(sums.to_host(), O.sums_grid(pts, ref, k, O.grid_scales(pts)))


@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -40, 2.0 ** 40, 2.0 ** 60])
def test_split_scales(gpu_ctx, scale):
    n, d, k = 8000, 6, 60
    pts = (clkmeans.generate_blobs(n, d, k, sigma=1.0, box=10.0, seed=3)[0] * np.float32(scale)).astype(np.float32)
    cen = np.ascontiguousarray(pts[:, :k])
    labels = zeros(n, np.uint32)
    gpu_ctx.labeling(gpu_ctx.config(clkmeans.STAGE_LABELING, "unroll_vector"), d, n, k, dev(pts), dev(cen), labels)
    hip.synchronize()
    np.testing.assert_array_equal(labels.to_host(), O.label(pts, cen))


@pytest.mark.parametrize("kind", ["blobs", "lattice", "offset", "special", "huge"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "n%d_d%d_k%d" % s)
def test_split_double(gpu_ctx, shape, kind):
    """Double points: labels and masses exact; sums within FP64 rounding of a
    different order (1e-13 of the cell's sum of |x|, as in test_gpu_f64)."""
    n, d, k = shape
    p32 = points(n, d, k, "blobs" if kind == "huge" else kind, n + d + k)
    cen32 = centroids(p32, k, kind)
    wiggle = np.random.default_rng(d).standard_normal(p32.shape) * 1e-9
    lattice = kind == "lattice"
    pts = p32.astype(np.float64) * (1.0 if lattice else 1.0 + wiggle)
    cen = np.ascontiguousarray(pts[:, np.arange(k) * 2 % n])
    if kind == "special":
        cen[~np.isfinite(cen)] = 1.0
        cen[~np.isfinite(cen32)] = cen32[~np.isfinite(cen32)]
    if kind == "huge":  # beyond FP32, and one centroid far beyond the others
        pts, cen = pts * 1e60, cen * 1e60
        cen[:, k - 1] *= 1e80
    ref = O.label_f64(pts, cen)
    labels = dev(np.full(n, 2 ** 64 - 1, np.uint64))
    gpu_ctx.labeling(gpu_ctx.config(clkmeans.STAGE_LABELING, "unroll_vector"), d, n, k, dev(pts), dev(cen), labels)
    hip.synchronize()
    np.testing.assert_array_equal(labels.to_host(), ref)
    labels = dev(np.full(n, 2 ** 64 - 1, np.uint64))
    sums, masses = zeros((d, k), np.float64), zeros(k, np.uint64)
    gpu_ctx.fused(gpu_ctx.config(clkmeans.STAGE_FUSED, "cluster_merge"), d, n, k, dev(pts), dev(cen), sums, labels, masses)
    hip.synchronize()
    np.testing.assert_array_equal(labels.to_host(), ref)
    np.testing.assert_array_equal(masses.to_host(), O.mass_u64(ref, k))
    if kind != "special":
        exact = O.sums_f64_dp(pts, ref, k)
        absx = np.stack([np.bincount(ref.astype(np.int64), weights=np.abs(x), minlength=k) for x in pts])
        assert np.all(np.abs(sums.to_host() - exact) <= 1e-13 * absx + 1e-300)


@pytest.mark.parametrize("n,d,k", [(100003, 3, 60), (100003, 4, 128), (20000, 7, 100), (20000, 16, 64), (20000, 24, 64), (20000, 48, 100)])
def test_double_centroids_between_two_halves(gpu_ctx, n, d, k):
    # coordinates whose FP32 rounding, scaled by a power of two, is exactly
    # between two FP16 values, while the double lies to one side: both parts
    # of the operand must come from the same rounding.  The points lie near
    # the planes between each centroid and its neighbour.
    rng = np.random.default_rng(d + k)
    cen = rng.uniform(1.0, 2.0, (d, k))
    cen = np.floor(cen * 1024) / 1024  # on the FP16 grid of [1, 2)
    cen += 2.0 ** -11  # between two of its values (the spacing is 2^-10)
    cen *= 1 + rng.choice([-1.0, 1.0], (d, k)) * 2.0 ** -27  # and a little off
    cen[0, 0] = 3.5
    a = rng.integers(0, k, n)
    other = cen[:, a]
    dist = ((cen[:, :, None] - cen[:, None, :]) ** 2).sum(0) + 1e9 * np.eye(k)
    near = dist.argmin(1)[a]
    t = 0.5 + rng.uniform(-1e-3, 1e-3, n)
    pts = np.ascontiguousarray(other * t + cen[:, near] * (1 - t))
    cfg = gpu_ctx.config(clkmeans.STAGE_LABELING, "unroll_vector")
    dl = zeros(n, np.uint64)
    gpu_ctx.labeling(cfg, d, n, k, dev(pts), dev(cen), dl)
    hip.synchronize()
    np.testing.assert_array_equal(dl.to_host(), O.label_f64(pts, np.ascontiguousarray(cen)))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,d,k", [(4101, 17, 290), (4164, 32, 129), (5000, 33, 200), (4099, 53, 290), (4097, 64, 300),
                                   (4100, 96, 100), (4097, 128, 90)])
def test_split_many_undecided(gpu_ctx, n, d, k, dtype):
    # far from the origin in every direction, two or more centroids close
    # together: most points stay undecided between a few of them.  Some points
    # and centroids that no score can order.
    rng = np.random.default_rng(n + d)
    centres = rng.uniform(-50, 50, (d, max(k // 3, 2)))
    pts = centres[:, rng.integers(0, centres.shape[1], n)] + rng.standard_normal((d, n)) * 0.3
    pts = np.ascontiguousarray(pts.astype(dtype))
    cen = np.ascontiguousarray(pts[:, :k])
    cen[:, k // 2] = cen[:, 1]  # ties
    cen[d - 1, k - 2] = np.nan
    pts[0, n - 1], pts[d // 2, n - 7], pts[0, 900] = np.nan, np.inf, 1e30
    f64 = dtype == np.float64
    ref = O.label_f64(pts, cen) if f64 else O.label(pts, cen)
    whole = np.uint64 if f64 else np.uint32
    dl = zeros(n, whole)
    gpu_ctx.labeling(gpu_ctx.config(clkmeans.STAGE_LABELING, "unroll_vector"), d, n, k, dev(pts), dev(cen), dl)
    hip.synchronize()
    np.testing.assert_array_equal(dl.to_host(), ref)
    if not f64 and d <= 32:
        dl, sums, masses = zeros(n, whole), zeros((d, k), np.float64), zeros(k, np.uint32)
        gpu_ctx.fused(gpu_ctx.config(clkmeans.STAGE_FUSED, "feature_sum"), d, n, k, dev(pts), dev(cen), sums, dl, masses)
        hip.synchronize()
        np.testing.assert_array_equal(dl.to_host(), ref)
        np.testing.assert_array_equal(masses.to_host(), O.mass(ref, k))
