"""The k-means work that this framework is used for, as cases that can be timed.

A case names an operation of onedal_amd.engine.Engine and its sizes:

  train        Engine.train          Lloyd training of dense rows
  infer        Engine.infer          labels (and the objective) of dense rows
  init         Engine.init_centroids k-means++ on dense rows
  csr_train    Engine.train_csr      Lloyd training of sparse rows
  csr_infer    Engine.infer_csr      labels and objective of sparse rows
  batch_train  Engine.train_batch_device   many independent trainings in one call
  batch_step   Engine.batch_step_device    one step of a continuous batch

Every operation is called as a program with its rows on the GPU calls it: one
Engine for the life of the program, CUDA tensors in, CUDA tensors out.
"""

import math
import random

import torch

from onedal_amd.engine import KM_INIT_PLUS_PLUS_DENSE, Engine

DEVICE = "cuda:0"
DTYPES = {"f32": torch.float32, "bf16": torch.float32, "f64": torch.float64}  # bf16: distances only
CHUNK = 1 << 20  # rows generated at a time

_engines = []


def _engine():
    """The program's engine (one context and its workspace)."""
    if not _engines:
        _engines.append(Engine(0))
    return _engines[0]


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one small request against a trained model: the call's latency
        dict(name="infer_tiny", op="infer", n=2000, d=20, k=10, dtype="f32", objective=True),
        # the plain Lloyd example: ten Gaussians, first-call size of most users
        dict(name="train_small", op="train", n=10_000, d=20, k=10, iters=50, thr=0.0, dtype="f32"),
        # the drop-in FP32 training workload
        dict(name="train_fp32", op="train", n=10_000_000, d=64, k=256, iters=20, thr=0.0, dtype="f32"),
        # the precision workload: BF16 distances with exact re-score
        dict(name="train_bf16", op="train", n=20_000_000, d=128, k=1024, iters=20, thr=0.0, dtype="bf16"),
        # a large inference request: new rows labelled once
        dict(name="infer_bf16", op="infer", n=5_000_000, d=128, k=512, dtype="bf16", objective=False),
        # float64 tables with an odd width, trained to a stop threshold
        dict(name="train_f64", op="train", n=300_007, d=50, k=100, iters=15, thr=1e-3, dtype="f64"),
        # float32 inference at odd sizes (rows not 16-byte aligned)
        dict(name="infer_ragged", op="infer", n=1_000_003, d=33, k=257, dtype="f32", objective=True),
        # wide rows (embeddings), beyond the matrix-core kernels' row registers
        dict(name="train_wide", op="train", n=100_000, d=512, k=256, iters=10, thr=0.0, dtype="f32"),
        # default initial centroids of the FP32 workload
        dict(name="init_plus_plus", op="init", n=10_000_000, d=64, k=256, dtype="f32"),
        # sparse rows, as the CSR benchmark
        dict(name="csr_train", op="csr_train", n=1_000_000, d=2000, k=256, nnz=20, ragged=False, base=0,
             iters=10, dtype="f32"),
        # many independent models in one call (one HIP graph)
        dict(name="batch_train", op="batch_train", count=128, n_lo=1000, n_hi=200_000, k_hi=128, mix=1, iters=20),
        # one step of a serving loop: a few jobs iterate, others get their final pass
        dict(name="batch_step", op="batch_step", count=8, n_lo=1000, n_hi=100_000, k_hi=128, mix=2, iters=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# most 2 n k d (passes) of a drawn dense case, by type and width: below the largest listed time
_FLOP_CAP = {"bf16": 4e13, "f32": 6e12, "f64": 2e12, "wide": 1e12}


def draw(rng):
    op = rng.choices(["train", "infer", "init", "csr_train", "csr_infer", "batch_train", "batch_step"],
                     [40, 20, 10, 8, 5, 9, 8])[0]
    if op in ("train", "infer", "init"):
        dtype = rng.choices(["f32", "bf16", "f64"], [45, 30, 25])[0]
        if op == "init" and dtype == "bf16":
            dtype = "f32"
        n, d, k = _log(rng, 1000, 20_000_000), _log(rng, 1, 1024), _log(rng, 2, 1024)
        if rng.random() < 0.5:
            d = max(4, d // 4 * 4)
        k = min(k, n // 2)
        iters = rng.randint(1, 50)
        n = min(n, int(2.5e9 / d) // (2 if dtype == "f64" else 1))
        passes = iters + 1 if op == "train" else 1
        cap = _FLOP_CAP["wide" if d > 256 else dtype] if op != "init" else 1e11
        while 2.0 * n * k * d * passes > cap:
            if passes > 4 and op == "train":
                iters = max(1, iters // 2)
                passes = iters + 1
            else:
                n //= 2
        # a call's row traffic, several sweeps of the rows each pass
        n = max(1000, min(n, int(1.2e10 / (d * passes))))
        k = min(k, n // 2)
        case = dict(op=op, n=n, d=d, k=k, dtype=dtype)
        if op == "train":
            case.update(iters=iters, thr=rng.choice([0.0, 0.0, 1e-3]))
        if op == "infer":
            case.update(objective=rng.random() < 0.5)
        return case
    if op in ("csr_train", "csr_infer"):
        d, k, nnz = _log(rng, 100, 4000), _log(rng, 4, 512), rng.randint(4, 60)
        iters = rng.randint(1, 10)
        n = min(_log(rng, 2000, 1_000_000), int(5e10 / (k * nnz * (iters + 1))))
        n = max(n, 2 * k)
        case = dict(op=op, n=n, d=d, k=k, nnz=min(nnz, d), ragged=rng.random() < 0.5, base=rng.randint(0, 1),
                    dtype=rng.choice(["f32", "f32", "f64"]))
        if op == "csr_train":
            case.update(iters=iters)
        return case
    count = _log(rng, 2, 128)
    return dict(op=op, count=count, n_lo=1000, n_hi=_log(rng, 5000, 200_000), k_hi=rng.randint(8, 128),
                mix=rng.randint(3, 1 << 20), iters=rng.randint(1, 20 if op == "batch_train" else 4))


def _mix(case):
    """(n, d, k) of each instance of a batched case: n log-uniform, d one of five
    widths, k uniform from 4."""
    rng = random.Random(case["mix"])
    return [(_log(rng, case["n_lo"], case["n_hi"]), rng.choice([8, 16, 32, 64, 128]), rng.randint(4, case["k_hi"]))
            for _ in range(case["count"])]


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _mixture(n, d, k, dtype, g, anisotropic=False):
    """Rows of a k-component Gaussian mixture, and the component centres."""
    reach = 50.0 if anisotropic else 10.0
    centres = (torch.rand((k, d), generator=g, device=DEVICE, dtype=dtype) * 2 - 1) * reach
    if anisotropic:
        scale = 10.0 ** (torch.rand((k, d), generator=g, device=DEVICE, dtype=dtype) * 2 - 1)
    else:
        scale = 0.5 + 1.5 * torch.rand((k, 1), generator=g, device=DEVICE, dtype=dtype)
    x = torch.empty((n, d), device=DEVICE, dtype=dtype)
    for r in range(0, n, CHUNK):
        part = x[r:r + CHUNK]
        lab = torch.randint(0, k, (part.shape[0],), generator=g, device=DEVICE)
        part.normal_(generator=g)
        part.mul_(scale[lab]).add_(centres[lab])
    return x, centres


def _rows(x, k, g):
    """k distinct random rows of x."""
    return x[torch.randperm(x.shape[0], generator=g, device=DEVICE)[:k]].clone()


def _sparse(case, g):
    """CSR rows: each holds the support columns of its cluster (some left out when
    ragged), values = the cluster's centre plus noise.  Also centroids: the first k
    rows to start a training from, or the clusters' centres to infer with."""
    n, d, k, m = case["n"], case["d"], case["k"], case["nnz"]
    dtype = DTYPES[case["dtype"]]
    support = torch.sort(torch.rand((k, d), generator=g, device=DEVICE).argsort(dim=1)[:, :m], dim=1).values
    level = torch.rand((k, m), generator=g, device=DEVICE, dtype=dtype) * 8 + 2
    truth = torch.randint(0, k, (n,), generator=g, device=DEVICE)
    cols = support[truth]
    vals = level[truth] + 0.3 * torch.randn((n, m), generator=g, device=DEVICE, dtype=dtype)
    if case["ragged"]:
        keep = torch.rand((n, m), generator=g, device=DEVICE) < 0.75
        length = keep.sum(1)
        cols, vals = cols[keep], vals[keep]
    else:
        length = torch.full((n,), m, device=DEVICE)
        cols, vals = cols.reshape(-1), vals.reshape(-1)
    offs = torch.zeros(n + 1, device=DEVICE, dtype=torch.int64)
    offs[1:] = torch.cumsum(length, 0)
    c = torch.zeros((k, d), device=DEVICE, dtype=dtype)
    if case["op"] == "csr_train":
        end = int(offs[k])
        row = torch.repeat_interleave(torch.arange(k, device=DEVICE), length[:k])
        c[row, cols[:end]] = vals[:end]
    else:
        c.scatter_(1, support, level)
        c += 0.05 * torch.rand((k, d), generator=g, device=DEVICE, dtype=dtype)
    return vals.contiguous(), cols.contiguous(), offs, c


def _batch(case, seed):
    g = _generator(seed)
    sets = []
    for n, d, k in _mix(case):
        x, centres = _mixture(n, d, k, torch.float32, g)
        sets.append((x, _rows(x, k, g), centres))
    return sets


def _views(flat, shapes):
    """Consecutive views of a flat tensor, one per shape."""
    got, at = [], 0
    for s in shapes:
        size = math.prod(s)
        got.append(flat[at:at + size].view(s))
        at += size
    return got


def _inputs(case, seed):
    op, g = case["op"], _generator(seed)
    if op.startswith("csr"):
        vals, cols, offs, c = _sparse(case, g)
        return dict(vals=vals, cols=cols + case["base"], offs=offs + case["base"], c=c)
    if op.startswith("batch"):
        return dict(sets=_batch(case, seed))
    x, centres = _mixture(case["n"], case["d"], case["k"], DTYPES[case["dtype"]], g, case["dtype"] == "bf16")
    if op == "train":
        return dict(x=x, c=_rows(x, case["k"], g))
    if op == "infer":  # a trained model's centroids: near the components' centres
        return dict(x=x, c=(centres + 0.05 * torch.randn(centres.shape, generator=g, device=DEVICE, dtype=x.dtype)))
    return dict(x=x)


def _split(case):
    """batch_step: how many of the jobs iterate (the others get their final pass)."""
    return max(1, case["count"] * 3 // 4)


def prepare(case, seed):
    state = dict(case=case, seed=seed, engine=_engine(), **_inputs(case, seed))
    if case["op"].startswith("batch"):
        # the caller's result buffers, one flat tensor each
        mix = _mix(case)
        step = _split(case) if case["op"] == "batch_step" else case["count"]
        labelled = mix if case["op"] == "batch_train" else mix[step:]
        state["centroids"] = torch.empty(sum(k * d for _, d, k in mix[:step]), device=DEVICE)
        state["labels"] = torch.empty(sum(n for n, _, _ in labelled), device=DEVICE, dtype=torch.int32)
        cs = _views(state["centroids"], [(k, d) for _, d, k in mix[:step]])
        ls = _views(state["labels"], [(n,) for n, _, _ in labelled])
        if case["op"] == "batch_train":
            state["xs"], state["c0s"] = [s[0] for s in state["sets"]], [s[1] for s in state["sets"]]
            state["outs"] = (cs, ls)
        else:
            state["iterated"] = [(x, c0, c) for (x, c0, _), c in zip(state["sets"], cs)]
            state["finished"] = [(x, m, None, l) for (x, _, m), l in zip(state["sets"][step:], ls)]
    torch.cuda.synchronize()  # the engine works on a stream of its own
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case, eng = state["case"], state["engine"]
    op = case["op"]
    if op == "train":
        c, labels, obj, iters = eng.train(state["x"], state["c"], case["iters"], case["thr"],
                                          bf16=case["dtype"] == "bf16")
        return dict(centroids=c, labels=labels, objective=obj, iterations=iters)
    if op == "infer":
        labels, obj = eng.infer(state["x"], state["c"], objective=case["objective"], bf16=case["dtype"] == "bf16")
        return dict(labels=labels, objective=obj)
    if op == "init":
        return dict(centroids=eng.init_centroids(state["x"], case["k"], KM_INIT_PLUS_PLUS_DENSE, state["seed"]))
    if op == "csr_train":
        c, labels, obj, iters = eng.train_csr(state["vals"], state["cols"], state["offs"], case["d"], state["c"],
                                              case["iters"], 0.0, base=case["base"])
        return dict(centroids=c, labels=labels, objective=obj, iterations=iters)
    if op == "csr_infer":
        labels, obj = eng.infer_csr(state["vals"], state["cols"], state["offs"], case["d"], state["c"],
                                    objective=True, base=case["base"])
        return dict(labels=labels, objective=obj)
    if op == "batch_train":
        _, _, objs, _ = eng.train_batch_device(state["xs"], state["c0s"], case["iters"], graph=True,
                                               outs=state["outs"])
    else:
        objs = eng.batch_step_device(state["iterated"], case["iters"], state["finished"])
    return dict(centroids=state["centroids"], labels=state["labels"],
                objectives=torch.tensor(objs, dtype=torch.float64))


def work(case):
    """Each pass over the rows (one per iteration and one for the final labels)
    reads them once and takes 2 k d operations a row; centroids and labels are
    written once."""
    op = case["op"]
    if op.startswith("batch"):
        mix, step = _mix(case), _split(case)
        n_bytes = n_flops = 0.0
        for i, (n, d, k) in enumerate(mix):
            passes = case["iters"] + 1 if op == "batch_train" else (case["iters"] if i < step else 1)
            n_bytes += passes * 4.0 * n * d + 4.0 * n + 8.0 * k * d
            n_flops += passes * 2.0 * n * k * d
        return dict(bytes=n_bytes, flops=n_flops)
    n, d, k = case["n"], case["d"], case["k"]
    size = 8 if case["dtype"] == "f64" else 4
    passes = case.get("iters", 0) + 1
    if op.startswith("csr"):
        stored = n * case["nnz"] * (0.75 if case["ragged"] else 1.0)
        return dict(bytes=passes * stored * (size + 8) + 8.0 * n + 2.0 * size * k * d + 4.0 * n,
                    flops=passes * 2.0 * stored * k)
    if op == "init":  # a step reads the rows and updates their distances
        return dict(bytes=(k - 1) * (float(size) * n * d + 16.0 * n), flops=(k - 1) * 3.0 * n * d)
    return dict(bytes=passes * float(size) * n * d + 2.0 * size * k * d + 4.0 * n, flops=passes * 2.0 * n * k * d)


# ---------------------------------------------------------------------------
# the same results in 64 bits, from plain torch
# ---------------------------------------------------------------------------
def _assign64(x, c):
    """Labels of rows x and their squared distances to centroids c."""
    labels = torch.empty(x.shape[0], device=x.device, dtype=torch.int64)
    dist = torch.empty(x.shape[0], device=x.device, dtype=torch.float64)
    cn = (c * c).sum(1)
    step = max(1, int(2.5e8) // c.shape[0])
    for r in range(0, x.shape[0], step):
        part = x[r:r + step].double()
        m = torch.addmm(cn, part, c.t(), alpha=-2.0).min(1)
        labels[r:r + step] = m.indices
        # the distance itself, without the cancellation of the expanded form
        dist[r:r + step] = (part - c[m.indices]).square_().sum(1)
    return labels, dist


def _means64(x, labels, c, dist):
    """Means of each cluster's rows; an empty cluster takes the row furthest from
    its centroid (the next furthest for the next empty one)."""
    k, d = c.shape
    copies = max(1, 65536 // k)  # partial sums, so that few rows add to the same address
    sums = torch.zeros((copies * k, d), device=x.device, dtype=torch.float64)
    for r in range(0, x.shape[0], 4 * CHUNK):
        lab = labels[r:r + 4 * CHUNK]
        at = torch.arange(lab.numel(), device=x.device) % copies
        sums.index_add_(0, at * k + lab, x[r:r + 4 * CHUNK].double())
    counts = torch.bincount(labels, minlength=k)
    new = sums.view(copies, k, d).sum(0) / counts.clamp(min=1).unsqueeze(1)
    empty = (counts == 0).nonzero().flatten()
    if empty.numel():
        new[empty] = x[torch.topk(dist, empty.numel()).indices].double()
    return new


def _train64(x, c0, iters, thr):
    c, prev, done = c0.double(), math.inf, 0
    while done < iters:
        labels, dist = _assign64(x, c)
        obj = float(dist.sum()) if thr > 0 else 0.0
        empty = int((torch.bincount(labels, minlength=c.shape[0]) == 0).sum()) if thr > 0 else 0
        if empty:
            obj -= float(torch.topk(dist, empty).values.sum())
        c = _means64(x, labels, c, dist)
        done += 1
        if thr > 0 and obj + thr > prev:
            break
        prev = obj
    return c, float(_assign64(x, c)[1].sum())


def _train_csr64(vals, cols, offs, d, c0, iters):
    vals, c = vals.double(), c0.double()
    n, k = offs.numel() - 1, c0.shape[0]
    rows = torch.sparse_csr_tensor(offs, cols, vals, size=(n, d))
    of_row = torch.repeat_interleave(torch.arange(n, device=vals.device), offs[1:] - offs[:-1])
    xs = torch.zeros(n, device=vals.device, dtype=torch.float64).index_add_(0, of_row, vals * vals)
    for done in range(iters + 1):
        m = ((c * c).sum(1) - 2.0 * (rows @ c.t())).min(1)
        closest = m.values + xs
        if done == iters:
            return c, float(closest.sum())
        copies = max(1, 4096 // k)
        sums = torch.zeros(copies * k * d, device=vals.device, dtype=torch.float64)
        sums.index_add_(0, ((of_row % copies) * k + m.indices[of_row]) * d + cols, vals)
        counts = torch.bincount(m.indices, minlength=k)
        c = sums.view(copies, k, d).sum(0) / counts.clamp(min=1).unsqueeze(1)
        empty = (counts == 0).nonzero().flatten().tolist()
        for j, r in zip(empty, torch.topk(closest, len(empty)).indices.tolist() if empty else []):
            c[j] = 0.0
            c[j, cols[offs[r]:offs[r + 1]]] = vals[offs[r]:offs[r + 1]]


def exact(case, seed):
    """Centroids and objectives.  Labels are whole numbers and have no value here,
    nor has a random choice of rows (init)."""
    op = case["op"]
    if op == "init":
        return None
    s = _inputs(case, seed)
    if op == "train":
        c, obj = _train64(s["x"], s["c"], case["iters"], case["thr"])
        return dict(centroids=c, labels=None, objective=obj, iterations=None)
    if op == "infer":
        if not case["objective"]:
            return None
        return dict(labels=None, objective=float(_assign64(s["x"], s["c"].double())[1].sum()))
    if op.startswith("csr"):
        c, obj = _train_csr64(s["vals"], s["cols"] - case["base"], s["offs"] - case["base"], case["d"], s["c"],
                              case.get("iters", 0))
        if op == "csr_infer":
            return dict(labels=None, objective=obj)
        return dict(centroids=c, labels=None, objective=obj, iterations=None)
    if op == "batch_train":
        got = [_train64(x, c0, case["iters"], 0.0) for x, c0, _ in s["sets"]]
        cs, objs = [c for c, _ in got], [o for _, o in got]
    else:
        step = _split(case)
        cs = []
        for x, c0, _ in s["sets"][:step]:
            c = c0.double()
            for _ in range(case["iters"]):
                labels, dist = _assign64(x, c)
                c = _means64(x, labels, c, dist)
            cs.append(c)
        objs = [float(_assign64(x, m.double())[1].sum()) for x, _, m in s["sets"][step:]]
    return dict(centroids=torch.cat([c.reshape(-1) for c in cs]), labels=None,
                objectives=torch.tensor(objs, dtype=torch.float64))
