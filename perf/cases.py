"""The work a user has this framework do, as timed cases.

Each case is one call (or one short sequence of calls) through the public
Python entry points: the single semiring products behind the drop-ins, the
FP16 emulation product, the repeated-squaring drivers, the two kNN paths and
the batched solver.  `listed()` names the cases, `draw()` makes more of the
same ranges, `prepare()` the inputs, `run()` one pass, `work()` what a pass
cannot do without and `exact()` its result in 64 bits.
"""
from __future__ import annotations

import math

import torch

import simd2_amd
from simd2_amd import graphs
from simd2_amd.batch import Batch
from simd2_amd.datasets import gaussian_clusters
from simd2_amd.knn import KnnBF16, knn_select, select_workspace_bytes
from simd2_amd.learned import converge_learned, load_model

FLOAT_OPS = ["min_plus", "plus_mul", "max_plus", "max_min", "max_mul", "min_mul", "min_max",
             "minus_square"]
GRAPH_OPS = ["min_plus", "max_min", "min_max"]
MIN_BASED = ("min_plus", "min_mul", "min_max")


def listed():
    return [
        # One tile's worth of work: what a call costs when the launch is the cost.
        {"name": "srgemm_min_plus_small", "kind": "srgemm", "op": "min_plus", "m": 96, "n": 80,
         "k": 64, "epilogue": True},
        # An ordinary product whose rows are not 16-byte aligned (the benchmark's off-grid shape).
        {"name": "srgemm_max_min_ragged", "kind": "srgemm", "op": "max_min", "m": 1000, "n": 777,
         "k": 300, "epilogue": False},
        # The suite's size for the semiring the headline names.
        {"name": "srgemm_min_plus_4096", "kind": "srgemm", "op": "min_plus", "m": 4096, "n": 4096,
         "k": 4096, "epilogue": True},
        # The suite's size for the one semiring that is a matrix product.
        {"name": "srgemm_plus_mul_4096", "kind": "srgemm", "op": "plus_mul", "m": 4096, "n": 4096,
         "k": 4096, "epilogue": True},
        # Boolean product in the reference's layout, one int32 per boolean.
        {"name": "orand_int32_4096", "kind": "orand", "m": 4096, "n": 4096, "k": 4096,
         "density": 0.02, "epilogue": True},
        # FP16 emulation product (the reference's tensor_srgemm).
        {"name": "emulation_min_plus_2048", "kind": "emulation", "op": "min_plus", "m": 2048,
         "n": 2048, "k": 2048, "epilogue": True},
        # All-pairs shortest paths of the benchmark's smallest application size.
        {"name": "apsp_1024", "kind": "closure", "op": "min_plus", "n": 1024, "p": 0.05},
        # Transitive closure of a sparse digraph at the application table's size.
        {"name": "gtc_8192", "kind": "reach", "n": 8192, "degree": 2.0},
        # Schedule-driven shortest paths on a road-like grid.
        {"name": "learned_grid_4096", "kind": "learned", "op": "min_plus", "family": "grid",
         "n": 4096, "degree": 0.0},
        # Nearest neighbours the reference's way: distance matrix, then top-k.
        {"name": "knn_direct_16384", "kind": "knn_direct", "q": 16384, "r": 16384, "dim": 128,
         "k": 16},
        # Nearest neighbours without the distance matrix.
        {"name": "knn_precision_16384", "kind": "knn_precision", "q": 16384, "r": 16384,
         "dim": 128, "k": 16},
        # A batch of small application graphs solved together.
        {"name": "batch_256", "kind": "batch", "count": 256, "nmin": 32, "nmax": 512,
         "sizes": 0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["srgemm", "srgemm", "srgemm", "orand", "emulation", "closure", "reach",
                       "learned", "knn_direct", "knn_precision", "batch"])
    if kind == "srgemm":
        return {"kind": kind, "op": rng.choice(FLOAT_OPS), "m": _log(rng, 16, 4096),
                "n": _log(rng, 16, 4096), "k": _log(rng, 16, 4096),
                "epilogue": rng.random() < 0.5}
    if kind == "orand":
        return {"kind": kind, "m": _log(rng, 64, 4096), "n": _log(rng, 64, 4096),
                "k": _log(rng, 64, 4096), "density": round(10 ** rng.uniform(-3, -0.5), 5),
                "epilogue": rng.random() < 0.5}
    if kind == "emulation":
        # the emulation takes multiples of 16 only
        return {"kind": kind, "op": rng.choice(FLOAT_OPS), "m": 16 * _log(rng, 1, 128),
                "n": 16 * _log(rng, 1, 128), "k": 16 * _log(rng, 1, 128),
                "epilogue": rng.random() < 0.5}
    if kind == "closure":
        n = _log(rng, 64, 2048)
        return {"kind": kind, "op": rng.choice(GRAPH_OPS), "n": n,
                "p": round(min(0.5, rng.uniform(4, 60) / n), 5)}
    if kind == "reach":
        return {"kind": kind, "n": _log(rng, 128, 8192), "degree": round(rng.uniform(0.5, 4), 3)}
    if kind == "learned":
        return {"kind": kind, "op": rng.choice(["min_plus", "max_min"]),
                "family": rng.choice(["er", "grid", "rgg"]), "n": _log(rng, 256, 4096),
                "degree": round(rng.uniform(8, 64), 2)}
    if kind in ("knn_direct", "knn_precision"):
        return {"kind": kind, "q": _log(rng, 512, 16384), "r": _log(rng, 1024, 16384),
                "dim": _log(rng, 16, 128), "k": rng.choice([1, 5, 10, 16, 16])}
    return {"kind": kind, "count": _log(rng, 16, 256), "nmin": 32, "nmax": rng.randint(64, 512),
            "sizes": rng.randint(1, 10 ** 6)}


# ---- inputs ------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _srgemm_values(op, shape, g):
    """The value ranges the operator meets: reliabilities in (0, 1] for the
    products of probabilities, features for the two sums, integer weights with
    missing edges for the rest."""
    if op in ("max_mul", "min_mul"):
        return 1.0 - torch.rand(shape, generator=g, device="cuda")
    if op in ("plus_mul", "minus_square"):
        return torch.randn(shape, generator=g, device="cuda")
    X = torch.randint(1, 101, shape, generator=g, device="cuda").float()
    hole = float("inf") if op in MIN_BASED else float("-inf")
    X[torch.rand(shape, generator=g, device="cuda") < 0.1] = hole
    return X


def _batch_graphs(case, seed):
    # the case fixes every graph's size and operator, the seed its edges
    specs = graphs.batch_specs(case["count"], case["sizes"], case["nmin"], case["nmax"])
    mats = [graphs.app_graph(torch, op, n, p, seed * 100003 + i)
            for i, (n, op, _, _, p, _) in enumerate(specs)]
    return specs, mats


def _learned_graph(case, seed):
    if case["family"] == "grid":
        return graphs.grid_family(torch, case["op"], case["n"], seed)
    if case["family"] == "rgg":
        return graphs.rgg_family(torch, case["op"], case["n"], case["degree"], seed)
    return graphs.er_family(torch, case["op"], case["n"], case["degree"] / case["n"], seed)


def _knn_points(case, seed):
    ref, centers = gaussian_clusters(torch, case["r"], case["dim"], 64, seed=2 * seed)
    query, _ = gaussian_clusters(torch, case["q"], case["dim"], 64, seed=2 * seed + 1,
                                 centers=centers)
    return ref, query


def _bits(shape, density, g):
    return (torch.rand(shape, generator=g, device="cuda") < density).int()


def prepare(case, seed):
    kind = case["kind"]
    g = _gen(seed)
    s = {"case": case}
    if kind == "srgemm":
        m, n, k = case["m"], case["n"], case["k"]
        s["A"] = _srgemm_values(case["op"], (m, k), g)
        s["B"] = _srgemm_values(case["op"], (k, n), g)
        s["C"] = _srgemm_values(case["op"], (m, n), g) if case["epilogue"] else None
        s["D"] = torch.empty((m, n), device="cuda")
    elif kind == "orand":
        m, n, k = case["m"], case["n"], case["k"]
        s["A"] = _bits((m, k), case["density"], g)
        s["B"] = _bits((k, n), case["density"], g)
        s["C"] = _bits((m, n), case["density"], g) if case["epilogue"] else None
        s["D"] = torch.empty((m, n), dtype=torch.int32, device="cuda")
    elif kind == "emulation":
        m, n, k = case["m"], case["n"], case["k"]
        s["A"] = _srgemm_values(case["op"], (m, k), g).half()
        s["B"] = _srgemm_values(case["op"], (k, n), g).half()
        s["C"] = _srgemm_values(case["op"], (m, n), g) if case["epilogue"] else None
        s["D"] = torch.empty((m, n), device="cuda")
    elif kind == "closure":
        s["graph"] = graphs.er_family(torch, case["op"], case["n"], case["p"], seed)
        s["X"], s["work"] = torch.empty_like(s["graph"]), torch.empty_like(s["graph"])
        s["flag"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif kind == "reach":
        n = case["n"]
        s["graph"] = _bits((n, n), case["degree"] / n, g)
        s["X"], s["work"] = torch.empty_like(s["graph"]), torch.empty_like(s["graph"])
        s["flag"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif kind == "learned":
        s["graph"] = _learned_graph(case, seed)
        s["X"] = torch.empty_like(s["graph"])
        s["model"] = load_model()[0]
        need = simd2_amd.learned._bind().simd2_converge_learned_workspace(case["n"], 64)
        s["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
    elif kind == "knn_direct":
        s["ref"], query = _knn_points(case, seed)
        s["query_t"] = query.t().contiguous()  # dimension-major, as the application holds it
        s["dist"] = torch.empty((case["r"], case["q"]), device="cuda")
        s["workspace"] = torch.empty(select_workspace_bytes(case["q"], case["r"], case["k"]),
                                     dtype=torch.uint8, device="cuda")
    elif kind == "knn_precision":
        s["ref"], s["query"] = _knn_points(case, seed)
        s["runner"] = KnnBF16(case["q"], case["r"], case["dim"])
    else:
        specs, s["mats"] = _batch_graphs(case, seed)
        s["batch"] = Batch([t[:4] for t in specs])
        # results go to one buffer per element type, each graph a view of it
        sizes = {torch.float32: 0, torch.int32: 0}
        places = []
        for X in s["mats"]:
            places.append(sizes[X.dtype])
            sizes[X.dtype] += X.numel()
        s["flat"] = {t: torch.empty(c, dtype=t, device="cuda") for t, c in sizes.items()}
        s["outs"] = [s["flat"][X.dtype][at:at + X.numel()].view(X.shape)
                     for X, at in zip(s["mats"], places)]
    return s


# ---- one pass ----------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "srgemm":
        return simd2_amd.srgemm(case["op"], s["A"], s["B"], s["C"], case["epilogue"], out=s["D"])
    if kind == "orand":
        return simd2_amd.srgemm("or_and", s["A"], s["B"], s["C"], case["epilogue"], out=s["D"])
    if kind == "emulation":
        return simd2_amd.tensor_srgemm(case["op"], s["A"], s["B"], s["C"], case["epilogue"],
                                       out=s["D"])
    if kind == "closure":
        # the driver works in place: the caller's graph is copied first
        s["X"].copy_(s["graph"])
        X, itr, _ = simd2_amd.converge(case["op"], s["X"], epilogue=case["op"] != "min_max",
                                       check="threshold", work=s["work"], flag=s["flag"])
        return X, itr
    if kind == "reach":
        s["X"].copy_(s["graph"])
        X, itr, _ = simd2_amd.converge("or_and", s["X"], work=s["work"], flag=s["flag"])
        return X, itr
    if kind == "learned":
        s["X"].copy_(s["graph"])
        X, itr, _, _, _ = converge_learned(case["op"], s["X"], s["model"],
                                           workspace=s["workspace"])
        return X, itr
    if kind == "knn_direct":
        simd2_amd.srgemm("minus_square", s["ref"], s["query_t"], out=s["dist"])
        return knn_select(s["dist"], case["k"], sqrt=True, workspace=s["workspace"])
    if kind == "knn_precision":
        return s["runner"](s["query"], s["ref"], case["k"], sqrt=True)
    b = s["batch"]
    for i, X in enumerate(s["mats"]):
        b.upload(i, X)
    b.solve()
    for i, out in enumerate(s["outs"]):
        b.download(i, out=out)
    itr, _ = b.iterations()
    return s["flat"][torch.float32], s["flat"][torch.int32], itr


# ---- what a pass cannot do without ---------------------------------------------


def work(case):
    """Bytes: inputs read once, outputs written once.  flops: one product and
    one sum per term; a closure is counted at the squarings that a path as
    long as the graph is deep needs (one more would only confirm it)."""
    kind = case["kind"]
    if kind in ("srgemm", "orand", "emulation"):
        m, n, k = case["m"], case["n"], case["k"]
        in_bytes = 2 if kind == "emulation" else 4
        return {"bytes": in_bytes * (m * k + k * n) + 4 * m * n * (2 if case["epilogue"] else 1),
                "flops": 2.0 * m * n * k}
    if kind in ("closure", "reach", "learned"):
        n = case["n"]
        squarings = {"closure": 3, "reach": 4, "learned": 4}[kind]
        return {"bytes": 8 * n * n, "flops": 2.0 * n ** 3 * squarings}
    if kind in ("knn_direct", "knn_precision"):
        q, r, d = case["q"], case["r"], case["dim"]
        return {"bytes": 4 * (q + r) * d + 8 * q * case["k"], "flops": 3.0 * q * r * d}
    # n uniform between nmin and nmax: second and third moments
    lo, hi, count = case["nmin"], case["nmax"], case["count"]
    span = max(hi - lo, 1)
    n2 = (hi ** 3 - lo ** 3) / (3 * span)
    n3 = (hi ** 4 - lo ** 4) / (4 * span)
    return {"bytes": 8 * count * n2, "flops": 2.0 * count * n3 * 0.8 * 4}


# ---- 64-bit results --------------------------------------------------------------


def _term(op, a, b):
    if op in ("min_plus", "max_plus"):
        return a + b
    if op in ("max_min",):
        return torch.minimum(a, b)
    if op in ("min_max",):
        return torch.maximum(a, b)
    if op == "minus_square":
        d = a - b
        return d * d
    return a * b


def _fold(op, x, y):
    if op in MIN_BASED:
        return torch.minimum(x, y)
    if op in ("plus_mul", "minus_square"):
        return x + y
    return torch.maximum(x, y)


def _identity(op):
    return math.inf if op in MIN_BASED else 0.0 if op in ("plus_mul", "minus_square") else -math.inf


def _product64(op, A, B, C, start):
    """fold over k of A[:, k] (x) B[k, :], the terms in the type of A and B,
    the fold in 64 bits, row block by row block."""
    m, k = A.shape
    n = B.shape[1]
    D = torch.empty((m, n), dtype=torch.float64, device=A.device)
    rows = max(1, min(m, (1 << 27) // max(n, 1)))
    deep = max(1, min(k, (1 << 25) // max(rows * n, 1)))
    for r in range(0, m, rows):
        acc = torch.full((min(rows, m - r), n), start, dtype=torch.float64, device=A.device)
        for q in range(0, k, deep):
            t = _term(op, A[r:r + rows, q:q + deep, None], B[None, q:q + deep, :]).double()
            t = (t.amin(1) if op in MIN_BASED else
                 t.sum(1) if op in ("plus_mul", "minus_square") else t.amax(1))
            acc = _fold(op, acc, t)
        D[r:r + rows] = acc
    return D if C is None else _fold(op, D, C.double())


def _closure64(op, X, epilogue):
    X = X.double()
    for _ in range(64):
        Y = _product64(op, X, X, X if epilogue else None, _identity(op))
        if torch.equal(X, Y):
            return X
        X = Y
    return X


def exact(case, seed):
    kind = case["kind"]
    if kind == "orand" or kind == "reach" or (kind == "learned" and case["n"] > 2048):
        return None  # whole numbers, or too many squarings for this plain form
    s = prepare(case, seed)
    if kind == "srgemm":
        op, A, B, C = case["op"], s["A"].double(), s["B"].double(), s["C"]
        if op == "plus_mul":
            D = A @ B
            return D if C is None else D + C.double()
        return _product64(op, A, B, C, _identity(op))
    if kind == "emulation":
        # the emulation rounds each term to FP16 and starts maxima at zero
        op = case["op"]
        start = 0.0 if op in ("max_plus", "max_min", "max_mul") else _identity(op)
        return _product64(op, s["A"], s["B"], s["C"], start)
    if kind == "closure":
        return _closure64(case["op"], s["graph"], case["op"] != "min_max"), None
    if kind == "learned":
        return _closure64(case["op"], s["graph"], True), None
    if kind == "batch":
        specs, mats = _batch_graphs(case, seed)
        done = [_closure64(op, X, epi).reshape(-1)
                for (_, op, epi, _, _, _), X in zip(specs, mats) if op != "or_and"]
        return torch.cat(done), None, None
    ref = s["ref"].double()
    query = (s["query"] if kind == "knn_precision" else s["query_t"].t()).double()
    parts = []
    for q in range(0, case["q"], 1024):
        block = query[q:q + 1024]
        near = (block.square().sum(1)[:, None] + ref.square().sum(1)[None, :]
                - 2.0 * block @ ref.t()).topk(case["k"], dim=1, largest=False).indices
        d2 = (block[:, None, :] - ref[near]).square().sum(2)
        parts.append(d2.sort(dim=1).values.sqrt())
    dist = torch.cat(parts)
    return (dist, None) if kind == "knn_precision" else (dist.t().contiguous(), None)
