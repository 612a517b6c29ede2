"""What users have this framework do, as cases that can be timed and compared.

A case is a dict of plain values; prepare() makes what a user's program holds before the call
(rows on the GPU or in host memory, a fitted model, device buffers of a serving loop), run() is
one call through the public entry points, the way a program makes it. The shapes are the
benchmark configurations of this repository, the two published examples of the estimator's
users and generic sizes round them; draw() gives more of the same ranges.
"""
import math

import numpy as np
import torch

from h2o4gpu_amd import KMeans
from h2o4gpu_amd.libs import kmeans_hip


def listed():
    return [
        # A serving loop labels a handful of requests per call with a small model: no
        # allocation, the caller's stream, nothing but launch latency.
        dict(name="serve_1k_d16_k8", kind="serve", dtype="float32", rows=1000, cols=16, k=8, data="blobs"),
        # A small table clustered at interactive speed: every iteration is a few microseconds.
        dict(name="fit_100k_d16_k8", kind="fit", dtype="float32", rows=100_000, cols=16, k=8, data="blobs",
             init="random", max_iter=20, tol=0.0),
        # The estimator as its documentation uses it: default start (k-means||) and default
        # tolerance, an ordinary table.
        dict(name="fit_default_1m_d64_k64", kind="fit", dtype="float32", rows=1_000_000, cols=64, k=64,
             data="blobs", init="k-means++", max_iter=50, tol=1e-4),
        # The headline shape: many short rows, a few hundred clusters, a fixed number of steps.
        dict(name="fit_10m_d32_k256", kind="fit", dtype="float32", rows=10_000_000, cols=32, k=256,
             data="blobs", init="random", max_iter=30, tol=0.0),
        # Colours of an image of ten million pixels (three 8-bit channels), as the estimator's
        # users quantise images: default start, run until the centres stand still.
        dict(name="fit_pixels_10m_d3_k27", kind="fit", dtype="float32", rows=10_116_514, cols=3, k=27,
             data="pixels", init="k-means++", max_iter=300, tol=1e-7),
        # A wide table of columns with scales of their own and a feature count that is no
        # multiple of anything: the shape of the published timing (261k x 298, 1000 clusters).
        dict(name="fit_table_261k_d298_k1000", kind="fit", dtype="float32", rows=261_117, cols=298, k=1000,
             data="table", init="random", max_iter=100, tol=0.0),
        # Double precision throughout, a model of a thousand wide rows.
        dict(name="fit_f64_2m_d256_k1024", kind="fit", dtype="float64", rows=2_000_000, cols=256, k=1024,
             data="blobs", init="random", max_iter=20, tol=0.0),
        # A visual codebook: long sparse 8-bit rows, thousands of clusters. (Rows without any
        # cluster structure: two correct float32 runs part at near-tie rows, and each further
        # step carries the difference to about four times as many labels; three steps keep them
        # comparable.)
        dict(name="fit_image_500k_d784_k4096", kind="fit", dtype="float32", rows=500_000, cols=784, k=4096,
             data="image", init="random", max_iter=3, tol=0.0),
        # Distances of held-out rows to every entry of such a codebook.
        dict(name="transform_100k_d784_k4096", kind="transform", dtype="float32", rows=100_000, cols=784,
             k=4096, data="image"),
        # Labelling new rows once against a fitted model: odd sizes on every axis.
        dict(name="predict_1m_d101_k500", kind="predict", dtype="float32", rows=1_000_003, cols=101, k=500,
             data="table"),
        # A wide table and a handful of clusters (segments of customers), one step after the other.
        dict(name="fit_500k_d784_k10", kind="fit", dtype="float32", rows=500_000, cols=784, k=10,
             data="table", init="random", max_iter=20, tol=0.0),
        # The whole reference-style call on host memory: fit, then predict on the same numpy rows
        # (colour quantisation of a photograph in double precision).
        dict(name="host_f64_273k_d3_k64", kind="host", dtype="float64", rows=273_280, cols=3, k=64,
             data="pixels", init="k-means++", max_iter=100, tol=1e-4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["serve", "fit", "fit", "fit", "predict", "predict", "transform", "host"])
    dtype = rng.choice(["float32", "float32", "float64"])
    if kind == "serve":
        cols, k = _log_int(rng, 3, 256), _log_int(rng, 2, 256)
        return dict(kind=kind, dtype=dtype, rows=_log_int(rng, 1000, 200_000), cols=cols, k=k, data="blobs")
    if kind == "host":
        return dict(kind=kind, dtype=dtype, rows=_log_int(rng, 20_000, 500_000), cols=_log_int(rng, 3, 64),
                    k=_log_int(rng, 2, 100), data=rng.choice(["blobs", "table"]),
                    init=rng.choice(["random", "k-means++"]), max_iter=rng.randint(10, 50), tol=1e-4)
    cols, k = _log_int(rng, 3, 800), _log_int(rng, 2, 4096)
    rows = _log_int(rng, 50_000, 10_000_000)
    # no dearer than the largest listed case: bounded rows, distances and matrix work
    steps = rng.randint(2, 6) if kind == "fit" else 1
    size = 8 if dtype == "float64" else 4
    rows = min(rows, int(4e9 / (cols * size)), int(8e12 / (2.0 * cols * k * steps)))
    if kind == "transform":
        rows = min(rows, int(3e9 / (k * size)))
    rows = max(rows, 40 * k)
    case = dict(kind=kind, dtype=dtype, rows=rows, cols=cols, k=k, data=rng.choice(["blobs", "table"]))
    if kind == "fit":
        case.update(init="random", max_iter=steps, tol=0.0)
    return case


def _rows(case, gen, rows):
    """Rows of the case's distribution on the GPU, in float32 and then in the case's type."""
    d, k, data = case["cols"], case["k"], case["data"]
    dev = "cuda"
    if data == "image":
        # sparse 8-bit rows: seven values in ten are zero
        X = torch.randint(1, 256, (rows, d), device=dev, generator=gen, dtype=torch.int16).float()
        X *= torch.rand((rows, d), device=dev, generator=gen) >= 0.7
    elif data == "pixels":
        # colours: soft blobs in the unit cube, 8 bits a channel
        base = torch.rand((max(8, k // 2), d), device=dev, generator=gen)
        lab = torch.randint(0, base.shape[0], (rows,), device=dev, generator=gen)
        X = base[lab] + 0.12 * torch.randn((rows, d), device=dev, generator=gen)
        X = (X.clamp_(0, 1) * 255).round_() / 255
    else:
        # clusters with overlapping tails; "table": columns of their own scale and offset
        centers = 20 * torch.rand((k, d), device=dev, generator=gen) - 10
        lab = torch.randint(0, k, (rows,), device=dev, generator=gen)
        X = torch.randn((rows, d), device=dev, generator=gen).mul_(2.0)
        X += centers[lab]
        if data == "table":
            scale = torch.exp(0.7 * torch.randn((1, d), device=dev, generator=gen))
            X.mul_(scale).add_(10 * scale * torch.randn((1, d), device=dev, generator=gen))
    return X.to(getattr(torch, case["dtype"]))


def _centres(case, X, gen):
    """Distinct rows of the data, each moved a little: centres as a fit would have left them."""
    pick = torch.randperm(X.shape[0], device="cuda", generator=gen)[:case["k"]]
    C = X[pick]
    C += 0.25 * X.std() * torch.randn(C.shape, device="cuda", generator=gen, dtype=C.dtype)
    return C.contiguous()


def _fitted(case, gen):
    """A fitted model, and rows of its distribution. (The fit has the centres for its rows, each
    the nearest to itself by far, so the model is these centres whatever the rounding.)"""
    X = _rows(case, gen, case["rows"])
    C = _centres(case, X, gen)
    model = KMeans(n_clusters=case["k"], init=C.cpu().numpy(), max_iter=1, tol=0.0, random_state=1)
    model.fit(C)
    return X, model, C


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000 + int(seed))
    kind = case["kind"]
    if kind == "serve":
        X = _rows(case, gen, case["rows"])
        C = X[torch.randint(0, X.shape[0], (case["k"],), device="cuda", generator=gen)].contiguous()
        labels = torch.empty(case["rows"], dtype=torch.int32, device="cuda")
        return dict(case=case, X=X, C=C, labels=labels, stream=torch.cuda.current_stream().cuda_stream)
    if kind == "fit":
        return dict(case=case, X=_rows(case, gen, case["rows"]), seed=int(seed) % 30000)
    if kind in ("predict", "transform"):
        X, model, _ = _fitted(case, gen)
        return dict(case=case, X=X, model=model)
    return dict(case=case, X=_rows(case, gen, case["rows"]).cpu().numpy(), seed=int(seed) % 30000)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "serve":
        kmeans_hip.predict_device_noalloc(np.dtype(case["dtype"]), case["rows"], case["cols"], case["k"],
                                          state["X"].data_ptr(), state["C"].data_ptr(),
                                          state["labels"].data_ptr(), state["stream"])
        return state["labels"]
    if kind == "predict":
        return state["model"].predict(state["X"])
    if kind == "transform":
        return state["model"].transform(state["X"])
    model = KMeans(n_clusters=case["k"], init=case["init"], max_iter=case["max_iter"], tol=case["tol"],
                   random_state=state["seed"])
    model.fit(state["X"])
    out = dict(centers=model.cluster_centers_, labels=model.labels_, inertia=model.inertia_)
    if kind == "host":
        out["predicted"] = model.predict(state["X"])
    return out


def exact(case, seed):
    """Distances (or the nearest centres) of the rows in float64; a fit has none: its start rows
    come from the framework's own random generator."""
    kind = case["kind"]
    if kind not in ("serve", "predict", "transform"):
        return None
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000 + int(seed))
    X = _rows(case, gen, case["rows"])
    if kind == "serve":
        C = X[torch.randint(0, X.shape[0], (case["k"],), device="cuda", generator=gen)]
    else:
        C = _centres(case, X, gen)
    C = C.double()
    cc = (C * C).sum(1)
    out = []
    step = max(1, int(2e8) // case["k"])
    for lo in range(0, X.shape[0], step):
        x = X[lo:lo + step].double()
        dist = torch.addmm((x * x).sum(1, keepdim=True) + cc, x, C.t(), alpha=-2.0).abs()
        out.append(dist if kind == "transform" else dist.argmin(1).to(torch.int32))
    return torch.cat(out)


def work(case):
    """Rows read once per pass over them, labels (or distances) written, 2 n k d operations per
    assignment pass (a fit of N updates makes N + 1 of them)."""
    n, d, k = case["rows"], case["cols"], case["k"]
    size = 8 if case["dtype"] == "float64" else 4
    passes = 1
    if case["kind"] == "fit":
        # (a run with a tolerance ends when it ends: a fifth of the bound is counted)
        passes = (case["max_iter"] if case["tol"] == 0.0 else max(2, case["max_iter"] // 5)) + 1
    elif case["kind"] == "host":
        passes = max(2, case["max_iter"] // 5) + 2
    out = n * k * size if case["kind"] == "transform" else 4 * n
    return {"bytes": float(passes * (n * d * size + 2 * k * d * size) + out),
            "flops": float(passes * 2.0 * n * k * d)}


def tolerance(case):
    """About four times what the float32 path differs by from the same call in float64, and from
    itself with the products of a distance summed in another order (both agree)."""
    f64 = case["dtype"] == "float64"
    if case["kind"] in ("serve", "predict"):
        # rows whose two nearest centres are a near-tie in the working precision
        return {"rel": 0.0, "differ": 1e-7 if f64 else 4e-5}
    if case["kind"] == "transform":
        return {"rel": 1e-13 if f64 else 8e-7, "max": 1e-12 if f64 else 7e-6}
    if f64:
        return {"rel": 1e-9, "max": 1e-6, "differ": 1e-6}
    if case["data"] == "image":
        # no cluster structure: near-tie rows of clusters of a hundred rows carry on
        return {"rel": 6e-3, "max": 0.7, "differ": 1e-2}
    return {"rel": 3e-3, "max": 0.25, "differ": 4e-3}
