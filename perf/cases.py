"""The workloads this library is measured on: clusterings through its public
entry points, from the smallest cloud to the largest data set.

Sizes, eps and minPts are those of hpdbscan_amd/datagen.py (the benchmark's
workloads), of bench.py's batched and serving legs and of the GPU tests.  Rows
are made on the GPU from the seed; every case of a kind keeps its sizes for
every seed, so that two seeds give two inputs of the same work.
"""
import math
import random

import numpy as np
import torch

from hpdbscan_amd import BORDER_MIN_CLUSTER, BORDER_ONE_THREAD, HPDBSCAN, Context, Server

DEVICE = "cuda:0"


def listed():
    return [
        # the smallest cloud of the batched workload, clustered by itself:
        # what a per-object loop over segmented point clouds calls
        {"name": "cloud_1k_3d", "kind": "cloud", "n": 1000, "d": 3, "dtype": "float32",
         "blobs": 12, "eps": 0.35, "min_points": 4, "border": "min"},
        # the reference's usual size: 100k rows in 3-D, device-resident
        {"name": "blobs_100k_3d", "kind": "cloud", "n": 100_000, "d": 3, "dtype": "float32",
         "blobs": 20, "eps": 0.3, "min_points": 4, "border": "min"},
        # the same size frame after frame in the same buffers: graph replay
        {"name": "replay_100k_3d", "kind": "replay", "n": 100_000, "d": 3, "dtype": "float32",
         "blobs": 20, "eps": 0.3, "min_points": 4, "border": "min"},
        # labels equal to the reference's run at one thread, ragged size, 2-D
        # (geographic points)
        {"name": "one_thread_300k_2d", "kind": "cloud", "n": 300_007, "d": 2, "dtype": "float32",
         "blobs": 30, "eps": 0.2, "min_points": 16, "border": "one_thread"},
        # the largest request of the serving workload, 4-D
        {"name": "cloud_5m_4d", "kind": "cloud", "n": 4_999_999, "d": 4, "dtype": "float32",
         "blobs": 25, "eps": 0.35, "min_points": 16, "border": "min"},
        # feature vectors in double precision, 6-D
        {"name": "features_30k_6d_f64", "kind": "cloud", "n": 30_011, "d": 6, "dtype": "float64",
         "blobs": 15, "eps": 0.5, "min_points": 8, "border": "min"},
        # quantised coordinates (an integer HDF5 data set), row-level union
        {"name": "lattice_200k_3d_i32", "kind": "cloud", "n": 200_003, "d": 3, "dtype": "int32",
         "blobs": 20, "eps": 30.0, "min_points": 8, "border": "min"},
        # the drop-in Python class on a host array: float64, host to host
        {"name": "drop_in_500k_3d", "kind": "host", "n": 500_009, "d": 3, "dtype": "float64",
         "blobs": 20, "eps": 0.2, "min_points": 8, "border": "min"},
        # the headline workload: 10M rows of anisotropic blobs
        {"name": "blobs_10m_3d", "kind": "aniso", "n": 10_000_000, "eps": 0.5, "min_points": 16},
        # the largest data set: 100M skewed 2-D rows (position fixes: hot
        # spots of millions of rows per cell, a few thousand strays)
        {"name": "skewed_100m_2d", "kind": "skewed", "n": 100_000_000, "eps": 0.01,
         "min_points": 32, "strays": 20_000},
        # thousands of clouds of 1k-200k rows in one batched call
        {"name": "batch_4096", "kind": "batch", "jobs": 4096, "n_min": 1000, "n_max": 200_000},
        # a burst of device-resident requests (10k-5M rows, 2-D to 4-D) on the
        # continuous-batching server
        {"name": "server_24", "kind": "server", "requests": 24, "n_min": 10_000,
         "n_max": 5_000_000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: every kind, its sizes log-uniform."""
    kind = rng.choice(["cloud", "cloud", "cloud", "cloud", "small", "small", "f64", "features",
                       "lattice", "one_thread", "replay", "host", "aniso", "skewed", "batch",
                       "server"])
    top = {"cloud": 5_000_000, "small": 30_000, "f64": 1_000_000, "features": 30_000,
           "lattice": 200_000, "one_thread": 300_000, "replay": 100_000, "host": 500_000}
    if kind in top:
        n = _log_int(rng, 10_000 if kind == "cloud" else 1000, top[kind])
        # blobs of 100 rows and more, so that small clouds have clusters too
        case = {"kind": "cloud", "n": n, "d": rng.choice([2, 3, 4]), "dtype": "float32",
                "blobs": rng.randint(5, max(5, min(50, n // 150))),
                "eps": round(rng.uniform(0.3 if n < 30_000 else 0.2, 0.5), 3),
                "min_points": rng.randint(4, 8 if n < 30_000 else 32), "border": "min"}
    if kind in ("cloud", "small"):
        return case
    if kind == "f64":
        return dict(case, dtype="float64")
    if kind == "features":
        return dict(case, d=rng.choice([5, 6]), dtype=rng.choice(["float32", "float64"]),
                    eps=round(rng.uniform(0.45, 0.6), 3))
    if kind == "lattice":
        return dict(case, d=rng.choice([2, 3]), dtype=rng.choice(["int16", "int32", "int64"]),
                    eps=float(rng.randint(20, 35)))
    if kind == "one_thread":
        return dict(case, border="one_thread")
    if kind == "replay":
        return dict(case, kind="replay")
    if kind == "host":
        return dict(case, kind="host", dtype="float64")
    if kind == "aniso":
        return {"kind": "aniso", "n": _log_int(rng, 1_000_000, 10_000_000),
                "eps": round(rng.uniform(0.4, 0.6), 3), "min_points": rng.randint(8, 24)}
    if kind == "skewed":
        return {"kind": "skewed", "n": _log_int(rng, 5_000_000, 100_000_000),
                "eps": round(rng.uniform(0.006, 0.01), 4), "min_points": rng.randint(32, 48),
                "strays": _log_int(rng, 5000, 20_000)}
    if kind == "batch":
        return {"kind": "batch", "jobs": _log_int(rng, 64, 4000), "n_min": 1000,
                "n_max": _log_int(rng, 10_000, 200_000)}
    return {"kind": "server", "requests": rng.randint(8, 24), "n_min": 10_000,
            "n_max": _log_int(rng, 500_000, 5_000_000)}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------

def _sizes(count, lo, hi):
    """`count` sizes, log-uniform over [lo, hi], in a fixed mixed order."""
    s = [int(round(lo * (hi / lo) ** ((i + 0.5) / count))) for i in range(count)]
    random.Random(count).shuffle(s)
    return s


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _rand(shape, g, dtype=torch.float32):
    return torch.rand(shape, generator=g, device=DEVICE, dtype=dtype)


def _randn(shape, g, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=dtype)


def _cloud(n, d, blobs, g, dtype=torch.float32):
    """Isotropic blobs (sigma 0.2, centres uniform in [0,10]^d) and 10 %
    uniform noise, in random order."""
    centres = 10.0 * _rand((blobs, d), g, dtype)
    x = centres[torch.randint(0, blobs, (n,), generator=g, device=DEVICE)]
    x += 0.2 * _randn((n, d), g, dtype)
    noise = _rand((n, 1), g) < 0.1
    return torch.where(noise, 10.0 * _rand((n, d), g, dtype), x).contiguous()


def _rows_of(case, g):
    dtype = getattr(torch, case["dtype"])
    if dtype.is_floating_point:
        return _cloud(case["n"], case["d"], case["blobs"], g, dtype)
    # a lattice of 0.01: coordinates 0-1000, sigma 20
    return torch.round(100.0 * _cloud(case["n"], case["d"], case["blobs"], g)).to(dtype)


def _aniso(n, g):
    """1000 anisotropic blobs in [0,100]^3 (per-axis sigma log-uniform in
    [0.1, 1], Dirichlet weights) and 5 % uniform noise."""
    k = 1000
    centres = 100.0 * _rand((k, 3), g)
    sigma = torch.exp(math.log(0.1) + (math.log(1.0) - math.log(0.1)) * _rand((k, 3), g))
    w = -torch.log1p(-_rand((k,), g, torch.float64))
    cum = torch.cumsum(w / w.sum(), 0)
    which = torch.searchsorted(cum, _rand((n,), g, torch.float64)).clamp_(max=k - 1)
    x = centres[which] + _randn((n, 3), g) * sigma[which]
    return torch.where(_rand((n, 1), g) < 0.05, 100.0 * _rand((n, 3), g), x).contiguous()


def _skewed(n, strays, g):
    """500 clusters in [0,1]^2 (log-normal sigma around 0.005, Zipf(1.2)
    weights) and `strays` uniform rows, too thin to be core by themselves."""
    k = 500
    centres = _rand((k, 2), g)
    sigma = torch.exp(math.log(0.005) + 0.7 * _randn((k,), g))
    w = torch.arange(1, k + 1, device=DEVICE, dtype=torch.float64) ** -1.2
    cum = torch.cumsum(w / w.sum(), 0).float()
    x = torch.empty((n, 2), device=DEVICE)
    step = 25_000_000
    for at in range(0, n, step):
        m = min(step, n - at)
        which = torch.searchsorted(cum, _rand((m,), g)).clamp_(max=k - 1)
        rows = (centres[which] + _randn((m, 2), g) * sigma[which, None]).clamp_(0.0, 1.0)
        x[at:at + m] = torch.where(_rand((m, 1), g) < strays / n, _rand((m, 2), g), rows)
    return x


def _batch(case, g):
    """The clouds of the batched workload one after the other: 5-50 blobs
    each, eps 0.2-0.5, minPts 4, 8 or 16."""
    sizes = _sizes(case["jobs"], case["n_min"], case["n_max"])
    jobs = len(sizes)
    counts = torch.tensor(sizes, device=DEVICE)
    job = torch.repeat_interleave(torch.arange(jobs, device=DEVICE), counts)
    blobs = torch.randint(5, 51, (jobs,), generator=g, device=DEVICE)
    centres = 10.0 * _rand((jobs * 50, 3), g)
    n = int(sum(sizes))
    which = (_rand((n,), g) * blobs[job]).long().clamp_(max=49)
    x = centres[job * 50 + which]
    del which, job
    x += 0.2 * _randn((n, 3), g)
    noise = _rand((n, 1), g) < 0.1
    x = torch.where(noise, 10.0 * _rand((n, 3), g), x).contiguous()
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    eps = (0.2 + 0.3 * _rand((jobs,), g)).cpu().numpy().astype(np.float32)
    pick = torch.randint(0, 3, (jobs,), generator=g, device=DEVICE).cpu().numpy()
    return x, offsets, eps, np.array([4, 8, 16], dtype=np.uint64)[pick]


def _request_shapes(case):
    return [(n, 2 + i % 3) for i, n in enumerate(_sizes(case["requests"], case["n_min"],
                                                        case["n_max"]))]


# --------------------------------------------------------------------------
# what a program keeps: one context per option, one server
# --------------------------------------------------------------------------
_kept = {}


def _context(border):
    if border not in _kept:
        _kept[border] = Context(0)
        _kept[border].set_border_rule(BORDER_ONE_THREAD if border == "one_thread"
                                      else BORDER_MIN_CLUSTER)
    return _kept[border]


def _server():
    if "server" not in _kept:
        _kept["server"] = Server(device=0)
    return _kept["server"]


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "server":
        rng = random.Random(seed)
        reqs = []
        for n, d in _request_shapes(case):
            x = _cloud(n, d, rng.randint(5, 50), g)
            reqs.append((x, rng.uniform(0.2, 0.5), rng.randint(4, 32),
                         torch.empty(n, dtype=torch.int64, device=DEVICE)))
        return {"kind": kind, "server": _server(), "requests": reqs}
    if kind == "host":
        return {"kind": kind, "model": HPDBSCAN(case["eps"], case["min_points"]),
                "x": _rows_of(case, g).cpu().numpy()}
    if kind == "batch":
        x, offsets, eps, min_points = _batch(case, g)
        return {"kind": kind, "ctx": _context("min"), "x": x, "offsets": offsets, "eps": eps,
                "min_points": min_points,
                "labels": torch.empty(len(x), dtype=torch.int64, device=DEVICE)}
    if kind == "aniso":
        x = _aniso(case["n"], g)
    elif kind == "skewed":
        x = _skewed(case["n"], case["strays"], g)
    else:
        x = _rows_of(case, g)
    if kind == "replay":
        ctx = Context(0)
        ctx.set_graph(True)
    else:
        ctx = _context(case.get("border", "min"))
    return {"kind": kind, "ctx": ctx, "x": x, "dtype": str(x.dtype).replace("torch.", ""),
            "eps": case["eps"], "min_points": case["min_points"],
            "labels": torch.empty(len(x), dtype=torch.int64, device=DEVICE)}


def run(state):
    kind = state["kind"]
    if kind == "server":
        server = state["server"]
        tickets = [server.submit_device(x.data_ptr(), x.shape[0], x.shape[1], np.float32, eps,
                                        min_points, labels.data_ptr())
                   for x, eps, min_points, labels in state["requests"]]
        for t in tickets:
            server.wait(t)
        return [labels for _, _, _, labels in state["requests"]]
    if kind == "host":
        return state["model"].cluster(state["x"], as_array=True)
    x, labels = state["x"], state["labels"]
    if kind == "batch":
        state["ctx"].cluster_batch_device(x.data_ptr(), state["offsets"], x.shape[1], np.float32,
                                          state["eps"], state["min_points"], labels.data_ptr())
    else:
        state["ctx"].cluster_device(x.data_ptr(), x.shape[0], x.shape[1], state["dtype"],
                                    state["eps"], state["min_points"], labels.data_ptr())
    return labels


def work(case):
    """Rows read once, int64 labels written once; the cell of every row."""
    kind = case["kind"]
    if kind == "batch":
        shapes = [(n, 3) for n in _sizes(case["jobs"], case["n_min"], case["n_max"])]
    elif kind == "server":
        shapes = _request_shapes(case)
    else:
        shapes = [(case["n"], {"aniso": 3, "skewed": 2}.get(kind) or case["d"])]
    size = torch.empty(0, dtype=getattr(torch, case.get("dtype", "float32"))).element_size()
    return {"bytes": sum(n * (d * size + 8) for n, d in shapes),
            "flops": sum(2 * n * d for n, d in shapes)}


def exact(case, seed):
    """Labels are whole numbers: there is no value to be nearer to."""
    return None
