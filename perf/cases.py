"""Performance cases of the search path: what is timed, on which inputs, and
what the results are compared with.

Each case is one call (or one training run) through the package's public
classes with inputs and outputs resident on the GPU, as a program that holds
its database in device memory makes it.  ``listed`` names the cases,
``draw`` makes others of the same ranges, ``prepare`` / ``run`` execute one,
``work`` states the bytes and operations it cannot do without, and ``exact``
evaluates it in 64 bits with plain torch.

Every result of this package is defined bit for bit (each distance is summed
in dimension order, ties go to the lower id or position), so the tolerance of
every case is ``"exact"``.
"""
from __future__ import annotations

import math

import torch

from vectorstorekit_amd import (HIPAccelerationEngine, HIPAcceleratorStrategy, IVFConfiguration,
                                IVFIndex, ProductQuantizer, ScalarQuantizer, SQ8Database,
                                VectorDatabase)
from vectorstorekit_amd.clustering import KMeansClustering, KMeansClusteringConfiguration

KSUB = 256

_accelerator = None


def _context():
    """The process's one device context, as an application opens it once."""
    global _accelerator
    if _accelerator is None:
        _accelerator = HIPAcceleratorStrategy(0)
    return _accelerator.initialize()


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # an interactive lookup: one query against a store of text embeddings
        {"name": "flat_single", "op": "flat", "n": 100_000, "d": 768, "nq": 1, "k": 10,
         "metric": "cosine", "data": "mixture"},
        # a small store and a small batch: launches and latency count
        {"name": "flat_small", "op": "flat", "n": 10_000, "d": 128, "nq": 100, "k": 10,
         "metric": "euclideanSquared", "data": "normal"},
        # a service's micro-batch over clustered embeddings, ragged sizes
        {"name": "flat_mid", "op": "flat", "n": 200_003, "d": 384, "nq": 333, "k": 50,
         "metric": "euclidean", "data": "mixture"},
        # the headline: an offline neighbour search over a million embeddings
        {"name": "flat_large", "op": "flat", "n": 1_000_000, "d": 768, "nq": 10_000, "k": 100,
         "metric": "cosineNormalized", "data": "normal"},
        # batchComputeDistances without topK: every distance is wanted
        {"name": "distances", "op": "distances", "n": 100_000, "d": 512, "nq": 32,
         "metric": "cosine", "data": "normal"},
        # one query through an IVF index of the default configuration
        {"name": "ivf_single", "op": "ivf", "n": 200_000, "d": 128, "nq": 1, "k": 10,
         "nlist": 1024, "nprobe": 10, "metric": "euclidean"},
        # a large query batch through a million-row IVF index
        {"name": "ivf_large", "op": "ivf", "n": 1_000_000, "d": 128, "nq": 10_000, "k": 10,
         "nlist": 4096, "nprobe": 32, "metric": "euclidean"},
        # the same index kept as product-quantized codes only
        {"name": "ivf_pq", "op": "ivf_codes", "kind": "pq", "n": 1_000_000, "d": 128, "M": 16,
         "nq": 10_000, "k": 10, "nlist": 4096, "nprobe": 32},
        # ten million int8 codes scanned for a thousand queries
        {"name": "sq8_large", "op": "sq8", "n": 10_000_000, "d": 128, "nq": 1000, "k": 100},
        # ten million PQ codes, the nearest thousand re-ranked on the rows
        {"name": "pq_large", "op": "pq", "n": 10_000_000, "M": 16, "dsub": 8, "nq": 1000,
         "k_adc": 1000, "k": 100, "rerank": "manhattan"},
        # product-quantizing a million rows for storage
        {"name": "pq_encode", "op": "pq_encode", "n": 1_000_000, "M": 16, "dsub": 8},
        # training an index's coarse centroids with the default seeding
        {"name": "kmeans_train", "op": "kmeans", "n": 100_000, "d": 128, "clusters": 1024,
         "iterations": 20, "init": "kMeansPlusPlus"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges; sizes spread over their logarithm,
    odd ones among them, each no dearer than the largest listed case."""
    op = rng.choice(["flat", "flat", "flat", "distances", "ivf", "ivf", "ivf_codes", "sq8", "pq",
                     "pq_encode", "kmeans"])
    if op == "flat":
        metric = rng.choice(["euclidean", "euclideanSquared", "cosine", "cosineNormalized",
                             "dotProduct", "manhattan"])
        n, d = _log(rng, 1000, 1_000_000), rng.choice([rng.randint(16, 1024), 96, 128, 384, 768])
        # Manhattan has no matrix form: its batches are smaller
        nq = max(1, min(_log(rng, 1, 10_000),
                        int((6e10 if metric == "manhattan" else 3e12) / (n * d))))
        return {"op": op, "n": n, "d": d, "nq": nq, "k": _log(rng, 1, 200), "metric": metric,
                "data": rng.choice(["normal", "mixture"])}
    if op == "distances":
        n, d = _log(rng, 1000, 200_000), rng.choice([rng.randint(16, 1024), 128, 512, 768])
        nq = max(1, min(_log(rng, 1, 256), int(2e10 / (n * d))))
        return {"op": op, "n": n, "d": d, "nq": nq, "data": "normal",
                "metric": rng.choice(["euclidean", "cosine", "dotProduct", "manhattan"])}
    if op in ("ivf", "ivf_codes"):
        nlist = _log(rng, 64, 4096)
        n = max(32 * nlist, _log(rng, 20_000, 1_000_000))
        nprobe = min(nlist, _log(rng, 1, 64))
        # (at most a quarter of the probed rows are asked for)
        k = min(_log(rng, 1, 100), nprobe * n // nlist // 4)
        if op == "ivf":
            d = rng.choice([rng.randint(16, 256), 96, 128, 768 if n <= 200_000 else 128])
            nq = max(1, min(_log(rng, 1, 10_000), int(3e10 * nlist / (nprobe * n * d))))
            return {"op": op, "n": n, "d": d, "nq": nq, "k": k, "nlist": nlist,
                    "nprobe": nprobe, "metric": rng.choice(["euclidean", "euclideanSquared"])}
        kind, M = rng.choice(["pq", "sq8"]), rng.choice([8, 16, 32])
        nq = max(1, min(_log(rng, 1, 10_000), int(3e8 * nlist / (nprobe * n))))
        return {"op": op, "kind": kind, "n": n, "d": M * rng.choice([4, 8]), "M": M, "nq": nq,
                "k": k, "nlist": nlist, "nprobe": nprobe}
    if op == "sq8":
        d = rng.choice([rng.randint(32, 512), 96, 128, 256])
        n = min(_log(rng, 10_000, 10_000_000), 1_280_000_000 // d)
        return {"op": op, "n": n, "d": d, "nq": _log(rng, 1, 1000), "k": _log(rng, 1, 100)}
    M, dsub = rng.choice([8, 16, 32]), rng.choice([4, 8])
    if op == "pq":
        n = _log(rng, 10_000, 10_000_000 * 128 // max(128, M * dsub))
        return {"op": op, "n": n, "M": M, "dsub": dsub, "nq": _log(rng, 1, 1000),
                "k_adc": _log(rng, 100, 1000), "k": _log(rng, 1, 100),
                "rerank": rng.choice(["manhattan", "euclidean", "none"])}
    if op == "pq_encode":
        return {"op": op, "n": _log(rng, 1000, 1_000_000), "M": M, "dsub": dsub}
    clusters = _log(rng, 16, 1024)
    return {"op": op, "n": max(8 * clusters, _log(rng, 5000, 200_000)),
            "d": rng.choice([rng.randint(16, 256), 96, 128]), "clusters": clusters,
            "iterations": rng.randint(3, 20), "init": rng.choice(["kMeansPlusPlus", "custom"])}


# ----------------------------------------------------------------- the inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _mixture(g, n, d, centres, nq):
    """Clustered rows and queries, as embeddings are: centres 2 N(0, I), each
    point its centre + 0.5 N(0, I)."""
    cent = 2.0 * torch.randn(centres, d, generator=g, device="cuda")
    a = torch.randint(0, centres, (n,), generator=g, device="cuda")
    x = cent[a].add_(torch.randn(n, d, generator=g, device="cuda"), alpha=0.5)
    b = torch.randint(0, centres, (nq,), generator=g, device="cuda")
    q = cent[b].add_(torch.randn(nq, d, generator=g, device="cuda"), alpha=0.5)
    return cent, x, q


def _code_books(x, M, dsub):
    """Codebooks from 256 rows, one codeword of every segment from each."""
    return x[:KSUB].reshape(KSUB, M, dsub).permute(1, 0, 2).contiguous()


def _encode(x, books):
    """PQ codes of the rows, by segment, in plain torch."""
    M, _, dsub = books.shape
    out = torch.empty(x.shape[0], M, dtype=torch.uint8, device=x.device)
    for s in range(0, x.shape[0], 1 << 20):
        c = x[s:s + (1 << 20)].to(books.dtype)
        for m in range(M):
            score = torch.addmm((books[m] * books[m]).sum(1), c[:, m * dsub:(m + 1) * dsub],
                                books[m].t(), alpha=-2.0)
            out[s:s + c.shape[0], m] = score.argmin(1).to(torch.uint8)
    return out


def _inputs(case, seed):
    """The case's tensors, from the seed alone."""
    g, op = _generator(seed), case["op"]
    if op in ("flat", "distances"):
        n, d, nq = case["n"], case["d"], case["nq"]
        if case["data"] == "mixture":
            _, x, q = _mixture(g, n, d, max(16, n // 1000), nq)
        else:
            x = torch.randn(n, d, generator=g, device="cuda")
            q = torch.randn(nq, d, generator=g, device="cuda")
        if case["metric"] == "cosineNormalized":
            x /= x.norm(dim=1, keepdim=True)
            q /= q.norm(dim=1, keepdim=True)
        return {"x": x, "q": q}
    if op in ("ivf", "ivf_codes"):
        cent, x, q = _mixture(g, case["n"], case["d"], case["nlist"], case["nq"])
        cent = cent + 0.1 * torch.randn(cent.shape, generator=g, device="cuda")
        got = {"x": x, "q": q, "centroids": cent}
        if case.get("kind") == "pq":
            got["books"] = _code_books(x, case["M"], case["d"] // case["M"])
        return got
    if op == "sq8":
        # what a per-dimension min/max quantizer makes of N(0, 1) rows
        def codes(rows):
            t = torch.randn(rows, case["d"], generator=g, device="cuda")
            return t.mul_(24.0).clamp_(-128, 127).to(torch.int8)
        return {"x": codes(case["n"]), "q": codes(case["nq"])}
    if op == "kmeans":
        cent, x, _ = _mixture(g, case["n"], case["d"], case["clusters"], 1)
        start = cent + 0.3 * torch.randn(cent.shape, generator=g, device="cuda")
        return {"x": x, "start": start}
    d = case["M"] * case["dsub"]
    _, x, q = _mixture(g, max(KSUB, case["n"]), d, 1024, case.get("nq", 1))
    return {"x": x, "q": q, "books": _code_books(x, case["M"], case["dsub"])}


class _State:
    def __init__(self, **kw):
        self.__dict__.update(kw)


def prepare(case, seed):
    ctx, t, op = _context(), _inputs(case, seed), case["op"]
    # the library's stream is its own: inputs are finished before it reads them
    torch.cuda.synchronize()
    if op == "flat":
        return _State(case=case, q=t["q"], db=VectorDatabase(ctx, t["x"]))
    if op == "distances":
        return _State(case=case, q=t["q"], db=VectorDatabase(ctx, t["x"]),
                      engine=HIPAccelerationEngine(ctx))
    if op in ("ivf", "ivf_codes"):
        cfg = IVFConfiguration(dimensions=case["d"], numberOfCentroids=case["nlist"],
                               numberOfProbes=case["nprobe"])
        idx = IVFIndex.build(ctx, cfg, t["centroids"].cpu().numpy(), t["x"])
        st = _State(case=case, q=t["q"], index=idx)
        if op == "ivf_codes":
            if case["kind"] == "pq":
                st.quantizer = ProductQuantizer(ctx, t["books"].cpu().numpy())
                idx.encodePQ(st.quantizer)
            else:
                st.quantizer = ScalarQuantizer(ctx, per_dim=True)
                st.quantizer.train(t["x"])
                idx.encodeSQ8(st.quantizer)
            idx.dropRows()
        return st
    if op == "sq8":
        return _State(case=case, q=t["q"], db=SQ8Database(ctx, t["x"]))
    if op == "pq":
        codes = _encode(t["x"], t["books"])
        torch.cuda.synchronize()
        pq = ProductQuantizer.upload(ctx, t["books"].cpu().numpy(), codes)
        rows = None if case["rerank"] == "none" else VectorDatabase(ctx, t["x"])
        return _State(case=case, q=t["q"], quantizer=pq, rows=rows)
    if op == "pq_encode":
        return _State(case=case, x=t["x"][:case["n"]].contiguous(),
                      quantizer=ProductQuantizer(ctx, t["books"].cpu().numpy()))
    cfg = KMeansClusteringConfiguration(maxIterations=case["iterations"], tolerance=1e-4,
                                        initMethod=case["init"], seed=int(seed),
                                        customCentroids=t["start"])
    return _State(case=case, x=t["x"], clustering=KMeansClustering(ctx, cfg))


# ------------------------------------------------------------------- the call

def run(state):
    case = state.case
    op = case["op"]
    if op == "flat":
        return state.db.search(state.q, case["k"], case["metric"])
    if op == "distances":
        return state.engine.batchComputeDistances(state.q, state.db, case["metric"])
    if op == "ivf":
        return state.index.search(state.q, case["k"], metric=case["metric"])
    if op == "ivf_codes":
        if case["kind"] == "pq":
            return state.index.searchPQ(state.q, case["k"])
        return state.index.searchSQ8(state.q, case["k"])
    if op == "sq8":
        return state.db.search(state.q, case["k"])
    if op == "pq":
        if case["rerank"] == "none":
            return state.quantizer.search(state.q, case["k"], k_adc=max(case["k"], case["k_adc"]))
        return state.quantizer.search(state.q, case["k"], k_adc=max(case["k"], case["k_adc"]),
                                      rerank_metric=case["rerank"], rerank_db=state.rows)
    if op == "pq_encode":
        return state.quantizer.encode(state.x)
    res = state.clustering.cluster(state.x, case["clusters"])
    return {"centroids": res.centroids, "assignments": res.assignments,
            "iterations": res.iterations, "inertia": res.inertia}


# ---------------------------------------------------------- work and tolerance

def work(case):
    op, n = case["op"], case["n"]
    if op == "flat":
        nq, d, k = case["nq"], case["d"], case["k"]
        return {"bytes": 4 * (n + nq) * d + 12 * nq * k, "flops": 2 * nq * n * d}
    if op == "distances":
        nq, d = case["nq"], case["d"]
        return {"bytes": 4 * ((n + nq) * d + nq * n), "flops": 2 * nq * n * d}
    if op in ("ivf", "ivf_codes"):
        nq, nlist, probe, k, d = (case["nq"], case["nlist"], case["nprobe"], case["k"], case["d"])
        pairs = nq * probe * n / nlist
        # the share of the lists that some query probes
        read = n * (1.0 - (1.0 - probe / nlist) ** nq)
        row, per_pair = 4 * d, 2 * d
        if op == "ivf_codes":
            row, per_pair = (case["M"], case["M"]) if case["kind"] == "pq" else (d, 2 * d)
        return {"bytes": int(read * row + 4 * (nlist + nq) * d + 12 * nq * k),
                "flops": int(2 * nq * nlist * d + pairs * per_pair)}
    if op == "sq8":
        nq, d = case["nq"], case["d"]
        return {"bytes": (n + nq) * d + 12 * nq * case["k"], "flops": 2 * nq * n * d}
    if op == "pq":
        nq, M, d = case["nq"], case["M"], case["M"] * case["dsub"]
        rows = 0 if case["rerank"] == "none" else min(n, nq * case["k_adc"])
        return {"bytes": n * M + 4 * rows * d + 4 * (nq + KSUB) * d + 12 * nq * case["k"],
                "flops": nq * n * M + 2 * nq * (KSUB + (case["k_adc"] if rows else 0)) * d}
    if op == "pq_encode":
        d = case["M"] * case["dsub"]
        return {"bytes": 4 * (n + KSUB) * d + n * case["M"], "flops": 2 * n * KSUB * d}
    d, c, it = case["d"], case["clusters"], case["iterations"]
    # the rows once per iteration; the seeding scores every row per centroid
    seeding = 1 if case["init"] == "kMeansPlusPlus" else 0
    return {"bytes": 4 * (n * d * (it + seeding) + 2 * c * d + n),
            "flops": 2 * n * c * d * (it + seeding)}


def tolerance(case):
    return "exact"


# ------------------------------------------------------------- 64-bit results

def _distances64(q, x, metric):
    """(queries, rows) distances in 64 bits."""
    if metric == "manhattan":
        return torch.cdist(q, x, p=1.0)
    if metric in ("euclidean", "euclideanSquared"):
        s = torch.addmm((x * x).sum(1), q, x.t(), alpha=-2.0)
        s = s.add_((q * q).sum(1, keepdim=True)).clamp_(min=0.0)
        return s.sqrt_() if metric == "euclidean" else s
    s = q @ x.t()
    if metric == "dotProduct":
        return s.neg_()
    if metric == "cosine":
        s /= q.norm(dim=1, keepdim=True) * x.norm(dim=1)[None, :] + 1e-8
    return s.neg_().add_(1.0)


def _nearest64(q, x, k, metric, convert=lambda t: t):
    """The k smallest distances of every query and their rows."""
    step_q = max(1, min(q.shape[0], 1024))
    step_x = max(1, int(2.5e8) // step_q)
    if metric == "manhattan":
        step_x = max(1, int(2e8) // step_q)
    dist, rows = [], []
    for a in range(0, q.shape[0], step_q):
        qa = q[a:a + step_q].double()
        bd = bi = None
        for s in range(0, x.shape[0], step_x):
            t = _distances64(qa, convert(x[s:s + step_x]), metric)
            v, i = torch.topk(t, min(k, t.shape[1]), dim=1, largest=False)
            i += s
            del t
            if bd is not None:
                v, i = torch.cat([bd, v], 1), torch.cat([bi, i], 1)
                v, p = torch.topk(v, min(k, v.shape[1]), dim=1, largest=False)
                i = i.gather(1, p)
            bd, bi = v, i
        dist.append(bd)
        rows.append(bi)
    return _padded(torch.cat(dist), k), torch.cat(rows)


def _padded(v, k, fill=float("inf")):
    return torch.nn.functional.pad(v, (0, k - v.shape[1]), value=fill) if v.shape[1] < k else v


def _probed64(case, t, score):
    """Smallest k of score(queries, rows, ids) over each query's probed lists."""
    cent, x, k = t["centroids"].double(), t["x"], case["k"]
    owner = torch.cat([_distances64(x[s:s + 65536].double(), cent, "euclidean").argmin(1)
                       for s in range(0, x.shape[0], 65536)])
    order = torch.argsort(owner, stable=True)
    size = torch.bincount(owner, minlength=case["nlist"])
    first = size.cumsum(0) - size
    out = []
    step = max(1, int(4e8 / (x.shape[1] * max(1.0, case["nprobe"] * x.shape[0] / case["nlist"]))))
    for a in range(0, t["q"].shape[0], step):
        q = t["q"][a:a + step].double()
        probes = torch.topk(_distances64(q, cent, "euclidean"), case["nprobe"], dim=1,
                            largest=False)[1]
        counts = size[probes].reshape(-1)
        ends = counts.cumsum(0)
        pair = torch.repeat_interleave(torch.arange(counts.numel(), device="cuda"), counts)
        rank = torch.arange(pair.numel(), device="cuda") - (ends - counts)[pair]
        ids = order[first[probes].reshape(-1)[pair] + rank]
        who = pair // case["nprobe"]
        total = size[probes].sum(1)
        col = torch.arange(pair.numel(), device="cuda") - (total.cumsum(0) - total)[who]
        table = torch.full((q.shape[0], max(k, int(total.max()))), float("inf"),
                           dtype=torch.float64, device="cuda")
        table[who, col] = score(q, who, ids)
        out.append(torch.topk(table, k, dim=1, largest=False)[0])
    return torch.cat(out)


def _decode64(codes, books):
    M = books.shape[0]
    return torch.cat([books[m][codes[:, m].long()] for m in range(M)], 1)


def exact(case, seed):
    t, op = _inputs(case, seed), case["op"]
    if op == "flat":
        v, _ = _nearest64(t["q"], t["x"], case["k"], case["metric"], lambda r: r.double())
        return v, None
    if op == "distances":
        return _distances64(t["q"].double(), t["x"].double(), case["metric"])
    if op == "ivf":
        def l2(q, who, ids):
            s = (q[who] - t["x"][ids].double()).square_().sum(1)
            return s.sqrt_() if case["metric"] == "euclidean" else s
        return _probed64(case, t, l2), None
    if op == "ivf_codes" and case["kind"] == "pq":
        books = t["books"].double()
        codes = _encode(t["x"], books)
        def adc(q, who, ids):
            return (q[who] - _decode64(codes[ids], books)).square_().sum(1).sqrt_()
        return _probed64(case, t, adc), None
    if op == "ivf_codes":
        low, high = t["x"].amin(0).double(), t["x"].amax(0).double()
        scale = 255.0 / (high - low)
        def code(v):
            return (v * scale - low * scale - 128.0).clamp_(-128, 127).trunc_()
        def dot(q, who, ids):
            return -(code(q)[who] * code(t["x"][ids].double())).sum(1)
        return -_probed64(case, t, dot), None
    if op == "sq8":
        v, _ = _nearest64(t["q"], t["x"], case["k"], "dotProduct", lambda r: r.double())
        return -v, None
    if op == "pq":
        books = t["books"].double()
        codes = _encode(t["x"], t["books"])
        k_adc = min(max(case["k"], case["k_adc"]), case["n"])
        v, rows = _nearest64(t["q"], codes, k_adc, "euclidean", lambda c: _decode64(c, books))
        if case["rerank"] != "none":
            v = torch.stack([_distances64(t["q"][i:i + 1].double(), t["x"][rows[i]].double(),
                                          case["rerank"])[0] for i in range(rows.shape[0])])
        v = torch.topk(v, min(case["k"], v.shape[1]), dim=1, largest=False)[0]
        return _padded(v, case["k"]), None
    if op == "pq_encode":
        return None
    if case["init"] == "kMeansPlusPlus":
        # each drawn centroid hangs on the rounding of all sums before it:
        # there is no 64-bit value of the seeding to compare with
        return None
    x, c = t["x"].double(), t["start"].double()
    before = math.inf
    for _ in range(case["iterations"]):
        near = [_distances64(x[s:s + 65536], c, "euclidean").min(1)
                for s in range(0, x.shape[0], 65536)]
        owner = torch.cat([v.indices for v in near])
        inertia = sum(v.values.sum().item() for v in near)
        size = torch.bincount(owner, minlength=case["clusters"])
        total = torch.zeros_like(c).index_add_(0, owner, x)
        c = torch.where(size[:, None] > 0, total / size.clamp(min=1)[:, None], c)
        if abs(inertia - before) < 1e-4:
            break
        before = inertia
    return {"centroids": c, "assignments": None, "iterations": None, "inertia": inertia}
