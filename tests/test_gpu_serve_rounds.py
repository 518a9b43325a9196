"""Serving rounds at their edges: jobs prepared together (one and several
slices of a row for the grid, NaN and infinity, rows of one to three values,
zero iterations) and singly once the round's buffer is full; tiles with four,
eight and sixteen waves; keep thresholds inside the finish and in the launch
of their own (k^2 d from 2^18), with centroid rows staged in LDS (d <= 32) and
not.  Each result equals the same job's alone, bit for bit, and the oracle's
Lloyd loop."""
import numpy as np
import pytest

import clkmeans
from clkmeans import hip
from oracle import oracle as O
from tests.test_gpu_serve import run_alone

pytestmark = pytest.mark.gpu

EDGES = [  # n, d, k
    (1, 3, 1), (3, 1, 2), (63, 4, 5), (1024, 5, 16), (1025, 8, 64), (4099, 9, 65), (5000, 16, 127), (5000, 16, 128),
    (3000, 17, 120), (3000, 32, 90), (3000, 32, 91), (2500, 32, 128), (2500, 40, 80), (2500, 64, 64), (2000, 3, 256),
    (65536, 2, 7), (65537, 3, 17), (140000, 4, 10),
]


def serve_and_check(ctx, specs, iters, labeling, special=(), zero=()):
    st = hip.Stream()
    reqs = []
    for i, (n, d, k) in enumerate(specs):
        rng = np.random.default_rng(1000 * i + n)
        pts = (rng.standard_normal((d, n)) * 3).astype(np.float32)
        if i in special:
            pts[0, n // 2], pts[d - 1, n // 3] = np.nan, np.inf
        cen = np.ascontiguousarray(pts[:, rng.integers(0, n, k)])
        reqs.append(clkmeans.ServeRequest(pts, cen, 0.0, max_iterations=0 if i in zero else iters, tolerance=0.0))
    b = clkmeans.Batch(ctx, max_jobs=len(specs), arena_bytes=256 << 20, max_d=64, max_k=512, labeling=labeling)
    for turn in range(2):  # the second call finds the first one's buffers
        for r in reqs:
            r.iterations = -1
        clkmeans.serve(b, reqs, st.handle)
        for i, r in enumerate(reqs):
            assert r.iterations == r.max_iterations
            if r.iterations == 0:
                np.testing.assert_array_equal(r.out_centroids.view(np.uint32), r.centroids.view(np.uint32))
                continue
            if turn == 0 and i not in special:
                _, rl, rm = O.lloyd(r.points, r.centroids, iters)
                np.testing.assert_array_equal(r.out_labels, rl)
                np.testing.assert_array_equal(r.out_masses, rm)
            c, l, m, _, shift = run_alone(ctx, r, st, labeling, max_d=64, max_k=512)
            np.testing.assert_array_equal(r.out_centroids.view(np.uint32), c.view(np.uint32))
            np.testing.assert_array_equal(r.out_labels, l)
            np.testing.assert_array_equal(r.out_masses, m)
    b.close()


@pytest.mark.parametrize("labeling", ["mfma_bf16", "unroll_vector"])
def test_round_edges(gpu_ctx, labeling):
    serve_and_check(gpu_ctx, EDGES, 4, labeling, special=(4, 9), zero=(2, 6))


def test_round_buffer_full(gpu_ctx):
    serve_and_check(gpu_ctx, [(600, 16, 512)] * 20, 2, "unroll_vector")
