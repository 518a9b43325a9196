"""Workloads of this library for timing: what a program has it do, through its
public entry points, over the sizes it is used at.

A case is one clustering (or one queue of clusterings) from its start to its
result:
  step         Lloyd iterations through the fused pass (Context.lloyd_step),
               points resident on the GPU
  three_stage  the same through the separate labeling, mass, centroid-update
               and divide operators
  serve        a queue of independent jobs through the batch engine
  run          a .conf-driven run over host arrays (kmeans_run)
Float points are float32 (uint32 labels and masses) or float64 (uint64).
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cl-kmeans_amd")


def _library():
    """The binding.  torch has brought its own HIP runtime into this process:
    the library and its hip module have to resolve to that one."""
    if "clkmeans" not in sys.modules:
        sys.path.insert(0, _PKG)
        before = os.environ.get("ROCM_PATH")
        if torch.version.hip and os.path.exists(os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so")):
            os.environ["ROCM_PATH"] = os.path.dirname(torch.__file__)
        try:
            import clkmeans
            clkmeans.load()
        finally:
            if before is None:
                os.environ.pop("ROCM_PATH", None)
            else:
                os.environ["ROCM_PATH"] = before
    return sys.modules["clkmeans"]


def _step(name, n, d, k, iters, strategy="cluster_merge", dtype="f32", track=False, sigma=1.0, box=50.0):
    return dict(name=name, kind="step", n=n, d=d, k=k, iters=iters, strategy=strategy, dtype=dtype, track=track,
                sigma=sigma, box=box)


def _three(name, n, d, k, iters, labeling="unroll_vector", mass="part_private", centroid="cluster_merge", dtype="f32",
           pin=False, sigma=1.0, box=50.0):
    return dict(name=name, kind="three_stage", n=n, d=d, k=k, iters=iters, labeling=labeling, mass=mass,
                centroid=centroid, dtype=dtype, pin=pin, sigma=sigma, box=box)


def listed():
    return [
        # a small table clustered to convergence, the shift watched: the time
        # is launches and latency
        _step("steps_small", 3000, 3, 5, 20, track=True, box=10.0),
        # the common size of the tuned configuration files: 2^20 points of 4
        # features, 10 clusters, 30 iterations
        _step("steps_1m", 1 << 20, 4, 10, 30),
        # the reference's own benchmark: 2 GiB of points, 30 iterations, with
        # the pass that keeps labels inside their keep radius
        _step("steps_2gib_bounded", 1 << 27, 4, 10, 30, strategy="cluster_merge_bounded"),
        # an odd number of rows, features that do not fill a power of two,
        # tens of overlapping clusters, the shift watched
        _step("steps_ragged", 2500003, 7, 33, 10, track=True, box=10.0),
        # wider rows (embeddings reduced to a few dozen features) through the
        # fused pass's other strategy
        _step("steps_wide", 700001, 24, 48, 10, strategy="feature_sum", box=5.0),
        # the three-stage configuration files' pipeline on a larger odd table
        _three("stages_10m", 10000019, 5, 20, 10, box=20.0),
        # quantisation to 256 entries of 32 features, plain FP32 labeling
        _three("stages_codebook", 400000, 32, 256, 5, mass="part_local", centroid="feature_sum", box=2.0),
        # the dense configuration: 64 features, 1024 clusters, labels from the
        # matrix cores, the points' operand copy kept by the program
        _three("stages_dense", 1 << 21, 64, 1024, 5, labeling="mfma_fp16", mass="part_local", pin=True, sigma=0.5,
               box=1.0),
        # the double / uint64 triple of the reference's benchmark
        _step("steps_double", 5000000, 4, 10, 10, dtype="f64"),
        # the double triple through the separate operators, wider rows
        _three("stages_double", 200003, 20, 64, 5, mass="part_local", centroid="feature_sum", dtype="f64", box=5.0),
        # 128 small clusterings that wait in a queue: sizes of the batched mix
        dict(name="serve_queue", kind="serve", jobs=128, log2n_max=16, labeling="mfma_bf16", sigma=1.0, box=10.0),
        # a whole run as a configuration file asks for it: host arrays in,
        # centroids, labels and masses out
        dict(name="conf_run", kind="run", pipeline="three_stage", n=1 << 20, d=4, k=10, iters=30, sigma=1.0, box=50.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _fit(n, d, k, iters, budget):
    """The most points (at most n) whose distance work stays in the budget."""
    return max(64, min(n, int(budget / (iters * (k * (2 * d + 3) + 4 * d + 40)))))


def draw(rng):
    kind = rng.choice(["step"] * 7 + ["three_stage"] * 5 + ["dense"] * 2 + ["f64_step", "f64_three"] * 2
                      + ["serve"] * 2 + ["run"])
    box = rng.choice([2.0, 5.0, 10.0, 20.0, 50.0])
    iters = rng.choice([5, 10, 20])
    if kind == "serve":
        return dict(kind="serve", jobs=_log_int(rng, 8, 128), log2n_max=rng.choice([12, 14, 16]),
                    labeling=rng.choice(["mfma_bf16", "mfma_fp16", "unroll_vector"]), sigma=1.0, box=box)
    n = _log_int(rng, 1 << 10, 1 << 25)
    d = _log_int(rng, 1, 64)
    k = max(2, min(_log_int(rng, 2, 512), n // 16))
    if kind == "run":
        d, k = min(d, 16), min(k, 64)
        n = _fit(min(n, 1 << 20), d, k, 30, 5e10)
        return dict(kind="run", pipeline=rng.choice(["single_stage", "three_stage"]), n=n, d=d, k=k, iters=30, sigma=1.0,
                    box=box)
    if kind == "step":
        c = _step("", _fit(n, d, k, iters, 1.2e11), d, k, iters, track=rng.random() < 0.5, box=box,
                  strategy=rng.choice(["cluster_merge", "cluster_merge", "feature_sum", "cluster_merge_bounded"]))
    elif kind == "three_stage":
        c = _three("", _fit(n, d, k, iters, 1.2e11), d, k, iters, box=box,
                   labeling=rng.choice(["unroll_vector", "unroll_vector", "unroll_vector_bounded"]),
                   mass=rng.choice(["global_atomic", "part_global", "part_local", "part_private"]),
                   centroid=rng.choice(["feature_sum", "feature_sum_pardim", "cluster_merge"]))
    elif kind == "dense":
        d, k, iters = rng.randint(24, 128), _log_int(rng, 64, 512), 5
        c = _three("", max(4096, _fit(n, d, k, iters, 1.5e11)), d, k, iters,
                   labeling=rng.choice(["mfma_fp16", "mfma_bf16"]), mass="part_local", pin=rng.random() < 0.5, sigma=0.5,
                   box=1.0)
    elif kind == "f64_step":
        d, k = min(d, 32), min(k, 128)
        c = _step("", _fit(n, d, k, iters, 3e10), d, k, iters, dtype="f64", track=rng.random() < 0.5, box=box,
                  strategy=rng.choice(["cluster_merge", "feature_sum"]))
    else:
        d, k = min(d, 32), min(k, 128)
        c = _three("", _fit(n, d, k, iters, 3e10), d, k, iters, dtype="f64", box=box, mass="part_local",
                   centroid="feature_sum")
    del c["name"]
    return c


class _Buffer:
    """A torch tensor as a device buffer of the binding."""

    def __init__(self, tensor, dtype):
        self.tensor, self.dtype, self.shape = tensor, np.dtype(dtype), tuple(tensor.shape)
        self.nbytes = tensor.numel() * tensor.element_size()

    def __int__(self):
        return self.tensor.data_ptr()

    @property
    def addr(self):
        return self.tensor.data_ptr()


def _blobs(n, d, k, sigma, box, seed, dtype):
    """Points [d][n]: normal noise around k centres, in random order."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 1)
    centres = (torch.rand(d, k, generator=g, device="cuda", dtype=dtype) * 2 - 1) * box
    blob = torch.randint(k, (n,), generator=g, device="cuda")
    pts = torch.empty(d, n, device="cuda", dtype=dtype)
    for f in range(d):
        pts[f] = centres[f][blob] + torch.randn(n, generator=g, device="cuda", dtype=dtype) * sigma
    return pts


def _dtype(case):
    return torch.float64 if case.get("dtype") == "f64" else torch.float32


def _queue(case, seed):
    """(n, d, k, points) of the queue's jobs: the batched mix's shapes are the
    same for every seed, the data are not."""
    specs = _library().job_mix(case["jobs"], seed=17, log2n=(10, case["log2n_max"]))
    return [(n, d, k, _blobs(n, d, k, case["sigma"], case["box"], int(seed) * 1009 + j, torch.float32))
            for j, (n, d, k, _) in enumerate(specs)]


def _conf(case):
    text = "[kmeans]\nclusters = %d\npipeline = %s\niterations = %d\n" % (case["k"], case["pipeline"], case["iters"])
    if case["pipeline"] == "single_stage":
        return text + "[kmeans.fused]\nstrategy = cluster_merge\n"
    return text + ("[kmeans.labeling]\nstrategy = unroll_vector\n[kmeans.mass_update]\nstrategy = part_private\n"
                   "[kmeans.centroid_update]\nstrategy = cluster_merge\n")


_TOL, _MAX_ITER = 1e-4, 50  # the served jobs' stopping rule


def prepare(case, seed):
    clkmeans = _library()
    if case["kind"] == "run":
        pts = _blobs(case["n"], case["d"], case["k"], case["sigma"], case["box"], seed, torch.float32).cpu().numpy()
        return dict(case=case, conf=_conf(case), points=pts, first=np.ascontiguousarray(pts[:, :case["k"]]))
    ctx = clkmeans.Context(0)
    if case["kind"] == "serve":
        return _prepare_queue(case, seed, ctx)
    n, d, k = case["n"], case["d"], case["k"]
    real = _dtype(case)
    f64 = real == torch.float64
    whole, np_whole, np_real = (torch.int64, np.uint64, np.float64) if f64 else (torch.int32, np.uint32, np.float32)
    pts = _blobs(n, d, k, case["sigma"], case["box"], seed, real)
    zeros = lambda shape, dtype: torch.zeros(shape, device="cuda", dtype=dtype)  # noqa: E731
    s = dict(case=case, ctx=ctx, f64=f64,
             points=_Buffer(pts, np_real),
             first=_Buffer(pts[:, :k].contiguous(), np_real),  # the first k points
             centroids=[_Buffer(zeros((d, k), real), np_real) for _ in range(2)],
             sums=_Buffer(zeros((d, k), torch.float64), np.float64),
             labels=_Buffer(zeros((n,), whole), np_whole),
             masses=_Buffer(zeros((k,), whole), np_whole),
             shift=_Buffer(zeros((1,), torch.float64), np.float64))
    if case["kind"] == "step":
        s["fused"] = ctx.config(clkmeans.STAGE_FUSED, case["strategy"])
    else:
        s["labeling"] = ctx.config(clkmeans.STAGE_LABELING, case["labeling"])
        s["mass"] = ctx.config(clkmeans.STAGE_MASS_UPDATE, case["mass"])
        s["update"] = ctx.config(clkmeans.STAGE_CENTROID_UPDATE, case["centroid"])
        if case["pin"]:
            ctx.labeling_pin_points(case["labeling"], d, n, s["points"])
    return s


def _prepare_queue(case, seed, ctx):
    clkmeans = _library()
    jobs = _queue(case, seed)
    flat = dict(centroids=np.zeros(sum(d * k for _, d, k, _ in jobs), np.float32),
                labels=np.zeros(sum(n for n, _, _, _ in jobs), np.uint32),
                masses=np.zeros(sum(k for _, _, k, _ in jobs), np.uint32))
    at = dict.fromkeys(flat, 0)

    def part(name, size):
        at[name] += size
        return flat[name][at[name] - size:at[name]]

    requests = []
    for n, d, k, pts in jobs:
        r = clkmeans.ServeRequest(_Buffer(pts, np.float32), np.ascontiguousarray(pts[:, :k].cpu().numpy()), 0.0,
                                  max_iterations=_MAX_ITER, tolerance=_TOL)
        r.out_centroids = part("centroids", d * k).reshape(d, k)
        r.out_labels, r.out_masses = part("labels", n), part("masses", k)
        requests.append(r)
    batch = clkmeans.Batch(ctx, max_jobs=case["jobs"], arena_bytes=1 << 30, max_d=32, max_k=256,
                           labeling=case["labeling"])
    return dict(case=case, ctx=ctx, batch=batch, requests=requests, flat=flat, stream=clkmeans.hip.Stream())


def run(s):
    clkmeans, case = _library(), s["case"]
    if case["kind"] == "run":
        cen, labels, masses, iters, _ = clkmeans.kmeans_run(s["conf"], s["points"], s["first"])
        return dict(centroids=cen, labels=labels, masses=masses, iterations=iters)
    if case["kind"] == "serve":
        clkmeans.serve(s["batch"], s["requests"], s["stream"])
        return dict(s["flat"], iterations=np.array([r.iterations for r in s["requests"]]))
    ctx, n, d, k = s["ctx"], case["n"], case["d"], case["k"]
    pts, sums, labels, masses = s["points"], s["sums"], s["labels"], s["masses"]
    if not s["f64"]:
        ctx.sum_grid_from_points(d, n, pts)  # once per data set, as the strategies do
    if "bounded" in case.get("strategy", "") or "bounded" in case.get("labeling", ""):
        ctx.fill_zero(labels)  # a fresh labels buffer
    old, new = s["first"], s["centroids"][0]
    shift = s["shift"] if case.get("track") else None
    for i in range(case["iters"]):
        if case["kind"] == "step":
            ctx.lloyd_step(s["fused"], d, n, k, pts, old, new, sums, labels, masses, max_shift=shift)
        else:
            ctx.labeling(s["labeling"], d, n, k, pts, old, labels)
            ctx.fill_zero(masses)
            ctx.fill_zero(sums)
            ctx.mass_update(s["mass"], n, k, labels, masses)
            ctx.centroid_update(s["update"], d, n, k, pts, sums, labels, masses)
            ctx.divide(d, k, sums, masses, new)
        old, new = new, s["centroids"][(i + 1) % 2]
    out = dict(centroids=old.tensor, sums=sums.tensor, labels=labels.tensor, masses=masses.tensor)
    if shift is not None:
        out["shift"] = shift.tensor
    return out


def work(case):
    if case["kind"] == "serve":
        # a dozen iterations to the stopping rule
        mix = _library().job_mix(case["jobs"], seed=17, log2n=(10, case["log2n_max"]))
        return {"bytes": sum(12 * n * (4 * d + 4) for n, d, k, _ in mix), "flops": sum(24 * n * d * k for n, d, k, _ in mix)}
    n, d, k, iters = case["n"], case["d"], case["k"], case["iters"]
    size = 8 if case.get("dtype") == "f64" else 4
    return {"bytes": iters * (n * size * (d + 1) + 2 * d * k * size), "flops": iters * 2 * n * d * k}


def _lloyd64(pts, cen, iters, tol=None):
    """Lloyd's iterations in 64 bits: (centroids, sums) [d][k] after `iters`
    iterations, or once no centroid moved by tol."""
    d, n = pts.shape
    k = cen.shape[1]
    cen = cen.double()
    chunk = max(1, (1 << 26) // k)
    ids = torch.arange(k, device=pts.device)
    for _ in range(iters):
        norm = (cen * cen).sum(0)
        sums = torch.zeros(d, k, device=pts.device, dtype=torch.float64)
        mass = torch.zeros(k, device=pts.device, dtype=torch.float64)
        for p in range(0, n, chunk):
            x = pts[:, p:p + chunk].double()
            dist = norm - 2.0 * (x.t() @ cen)
            dist = torch.where(dist.isnan(), torch.inf, dist)
            hot = (dist.argmin(1, keepdim=True) == ids).double()
            sums += x @ hot
            mass += hot.sum(0)
        new = sums / mass
        move = (new - cen).square().sum(0).sqrt()
        cen = new
        if tol is not None and float(move[mass > 0].max()) < tol:
            break
    return cen, sums


def exact(case, seed):
    if case["kind"] == "serve":
        cen = [_lloyd64(pts, pts[:, :k], _MAX_ITER, _TOL)[0].reshape(-1) for _, _, k, pts in _queue(case, seed)]
        return dict(centroids=torch.cat(cen), labels=None, masses=None, iterations=None)
    pts = _blobs(case["n"], case["d"], case["k"], case["sigma"], case["box"], seed, _dtype(case))
    cen, sums = _lloyd64(pts, pts[:, :case["k"]], case["iters"])
    if case["kind"] == "run":
        return dict(centroids=cen, labels=None, masses=None, iterations=None)
    out = dict(centroids=cen, sums=sums, labels=None, masses=None)
    if case.get("track"):
        out["shift"] = None
    return out
