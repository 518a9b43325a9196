"""Captured operators.  Those that need no scratch memory of their own (the
global-atomic mass update, the centroid update of many clusters) are captured
into a graph on a context that has none yet, where growing it would break the
capture; a graph of one MFMA labeling, whose replays hand the score offset on.
Every replay gives the eager result, with the program's own eager work
between."""
import ctypes

import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.helpers import dev, zeros

pytestmark = pytest.mark.gpu


class Graph:
    """What fn enqueues on a stream, captured."""

    def __init__(self, fn):
        L = hip.lib()
        self.L, self.stream = L, hip.Stream()
        self.graph, self.exec = ctypes.c_void_p(), ctypes.c_void_p()
        hip.synchronize()
        hip.check(L.hipStreamBeginCapture(self.stream.handle, 0), "begin capture")
        try:
            fn(self.stream.handle)
        finally:
            rc = L.hipStreamEndCapture(self.stream.handle, ctypes.byref(self.graph))
        hip.check(rc, "end capture")
        hip.check(L.hipGraphInstantiate(ctypes.byref(self.exec), self.graph, None, None, ctypes.c_size_t(0)), "instantiate")

    def launch(self):
        hip.check(self.L.hipGraphLaunch(self.exec, self.stream.handle), "launch")
        self.stream.synchronize()

    def close(self):
        self.L.hipGraphExecDestroy(self.exec)
        self.L.hipGraphDestroy(self.graph)


@pytest.mark.parametrize("n,k", [(1000, 5), (700001, 36), (3000000, 4000)])
def test_global_atomic_masses(n, k):
    ctx = clkmeans.Context(0)
    rng = np.random.default_rng(n)
    masses, dl = zeros(k, np.uint32), dev(rng.integers(0, k, n).astype(np.uint32))
    cfg = ctx.config(clkmeans.STAGE_MASS_UPDATE, "global_atomic")
    g = Graph(lambda st: ctx.mass_update(cfg, n, k, dl, masses, stream=st))
    for turn in range(3):
        lab = rng.integers(0, k, n).astype(np.uint32)
        dl.copy_from(lab)
        ctx.fill_zero(masses)
        hip.synchronize()
        g.launch()
        np.testing.assert_array_equal(masses.to_host(), np.bincount(lab, minlength=k))
    g.close()
    ctx.close()


@pytest.mark.parametrize("n,d,k", [(40000, 6, 5000), (100001, 5, 9000), (3000, 5, 30), (200000, 8, 300)])
def test_centroid_update(n, d, k):
    ctx = clkmeans.Context(0)
    rng = np.random.default_rng(n)
    pts = rng.standard_normal((d, n)).astype(np.float32)
    dp, dl, sums = dev(pts), dev(rng.integers(0, k, n).astype(np.uint32)), zeros((d, k), np.float64)
    ctx.sum_grid_from_points(d, n, dp)
    hip.synchronize()
    cfg = ctx.config(clkmeans.STAGE_CENTROID_UPDATE, "cluster_merge")
    g = Graph(lambda st: ctx.centroid_update(cfg, d, n, k, dp, sums, dl, stream=st))
    for turn in range(3):
        lab = rng.integers(0, k, n).astype(np.uint32)
        dl.copy_from(lab)
        ctx.fill_zero(sums)
        hip.synchronize()
        g.launch()
        np.testing.assert_array_equal(sums.to_host(), O.sums_grid(pts, lab, k, O.grid_scales(pts)))
    g.close()
    ctx.close()


@pytest.mark.parametrize("strategy", ["mfma_fp16", "mfma_bf16"])
@pytest.mark.parametrize("warm", [1, 2])
def test_mfma_labeling(strategy, warm):
    n, d, k = 30000, 40, 100
    ctx = clkmeans.Context(0)
    pts, _ = clkmeans.generate_blobs(n, d, k, sigma=1.0, box=3.0, seed=5)
    cen = np.ascontiguousarray(pts[:, :k])
    dp, dc, dl = dev(pts), dev(cen), zeros(n, np.uint32)
    cfg = ctx.config(clkmeans.STAGE_LABELING, strategy)
    for _ in range(warm):  # the scratch memory
        ctx.labeling(cfg, d, n, k, dp, dc, dl)
    g = Graph(lambda st: ctx.labeling(cfg, d, n, k, dp, dc, dl, stream=st))
    for scale in (1.0, 50.0, 0.01, 1.0):  # the offset of one replay does not fit the next one's data
        p = (pts * np.float32(scale)).astype(np.float32)
        c = np.ascontiguousarray(p[:, :k])
        dp.copy_from(p)
        dc.copy_from(c)
        for _ in range(2):
            hip.synchronize()
            g.launch()
            np.testing.assert_array_equal(dl.to_host(), O.label(p, c))
        ctx.labeling(cfg, d, n, k, dp, dc, dl)
    g.close()
    ctx.close()
