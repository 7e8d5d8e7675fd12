"""The work this package is used for, as cases that can be timed and compared.

Each case goes through the public Python mirror (`proxima_amd`), as a program
that holds an index, a set of points or a batch of queries would call it:

- `flat`: exact search of a FlatIndex (all MFMA metrics, host or device
  queries, filters, removed rows);
- `sq8`: search of an Sq8Index, with and without rescoring;
- `ivfpq`: search of a trained IvfPqIndex, with and without rerank;
- `ivfpq_train`: training an IvfPqIndex on the vectors it holds (coarse
  k-means, residual product quantizer, encoding of every vector);
- `kmeans`: k-means++ and Lloyd on device-resident points, or Lloyd from given
  centroids.

Every result of these paths is defined to the bit (exact distances in a fixed
operation order, ties by id, seeded training), so `tolerance` is "exact".
"""
import math

import numpy as np
import torch

import proxima_amd as px

DEV = "cuda:0"
METRICS = {"euclidean": px.Metric.EUCLIDEAN, "cosine": px.Metric.COSINE, "inner_product": px.Metric.INNER_PRODUCT}


def listed():
    return [
        # an interactive lookup: one query from host memory, answered at once
        {"name": "flat_one_query", "kind": "flat", "metric": "euclidean", "n": 100_000, "dim": 128, "nq": 1, "k": 10,
         "host": True, "accept": 1.0, "removed": 0},
        # a server that gathers a few requests before it searches
        {"name": "flat_few_queries", "kind": "flat", "metric": "euclidean", "n": 100_000, "dim": 128, "nq": 48,
         "k": 10, "host": False, "accept": 1.0, "removed": 0},
        # a batch over a small corpus (the 100k x 128 benchmark)
        {"name": "flat_batch", "kind": "flat", "metric": "euclidean", "n": 100_000, "dim": 128, "nq": 1000, "k": 10,
         "host": False, "accept": 1.0, "removed": 0},
        # a batch over a large corpus of wide embeddings (the headline benchmark)
        {"name": "flat_wide", "kind": "flat", "metric": "cosine", "n": 1_000_000, "dim": 768, "nq": 1024, "k": 10,
         "host": False, "accept": 1.0, "removed": 0},
        # long result lists under a filter, over a store with holes, nothing a multiple of a tile
        {"name": "flat_filtered", "kind": "flat", "metric": "inner_product", "n": 300_007, "dim": 300, "nq": 313,
         "k": 100, "host": False, "accept": 0.5, "removed": 57},
        # byte codes of a large corpus (the 10M x 96 benchmark)
        {"name": "sq8_batch", "kind": "sq8", "metric": "inner_product", "n": 10_000_000, "dim": 96, "nq": 1024,
         "k": 10, "rescore": 0, "host": False},
        # byte codes with exact-query rescoring, a few host queries, odd sizes
        {"name": "sq8_rescored", "kind": "sq8", "metric": "cosine", "n": 1_000_003, "dim": 100, "nq": 33, "k": 20,
         "rescore": 100, "host": True},
        # compressed search of a large corpus (the 10M x 128 benchmark)
        {"name": "ivfpq_batch", "kind": "ivfpq", "metric": "euclidean", "n": 10_000_000, "dim": 128, "nlist": 4096,
         "subspaces": 16, "nprobe": 32, "rerank": 0, "nq": 1024, "k": 10, "host": False},
        # compressed search whose best candidates are rescored exactly, a small host batch
        {"name": "ivfpq_rerank", "kind": "ivfpq", "metric": "cosine", "n": 500_000, "dim": 96, "nlist": 1024,
         "subspaces": 12, "nprobe": 16, "rerank": 100, "nq": 100, "k": 10, "host": True},
        # building the compressed index
        {"name": "ivfpq_train", "kind": "ivfpq_train", "metric": "euclidean", "n": 300_000, "dim": 96, "nlist": 1024,
         "subspaces": 12},
        # a large clustering from its seed (the 2M x 128 benchmark)
        {"name": "kmeans_large", "kind": "kmeans", "n": 2_000_000, "dim": 128, "clusters": 4096, "iterations": 10,
         "given": False},
        # refining a small clustering from given centroids, odd sizes
        {"name": "kmeans_small", "kind": "kmeans", "n": 60_011, "dim": 100, "clusters": 300, "iterations": 8,
         "given": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flat", "flat", "flat", "sq8", "ivfpq", "ivfpq_train", "kmeans", "kmeans"])
    if kind == "flat":
        dim = rng.choice([_log(rng, 16, 768), rng.choice([64, 96, 128, 256, 384, 768])])
        n = _log(rng, 5_000, min(1_000_000, 400_000_000 // dim))
        nq = _log(rng, 1, 1024)
        host = rng.random() < 0.4
        accept = 1.0 if host else rng.choice([1.0, round(rng.uniform(0.1, 0.9), 2)])  # masks come with device queries
        return {"kind": kind, "metric": rng.choice(sorted(METRICS)), "n": n, "dim": dim, "nq": nq,
                "k": rng.choice([1, 10, _log(rng, 2, 100)]), "host": host, "accept": accept,
                "removed": rng.choice([0, 0, 31])}
    if kind == "sq8":
        return {"kind": kind, "metric": rng.choice(["cosine", "inner_product"]), "n": _log(rng, 50_000, 4_000_000),
                "dim": rng.choice([64, 96, 128, rng.randint(33, 256)]), "nq": _log(rng, 1, 1024),
                "k": _log(rng, 1, 100), "rescore": rng.choice([0, 0, 100]), "host": rng.random() < 0.4}
    if kind in ("ivfpq", "ivfpq_train"):
        m = rng.choice([8, 12, 16, 16, 24])
        dim = m * rng.choice([4, 6, 8])
        nlist = _log(rng, 64, 2048)
        c = {"kind": kind, "metric": rng.choice(["cosine", "euclidean"]), "n": _log(rng, 60_000, 1_000_000),
             "dim": dim, "nlist": nlist, "subspaces": m}
        if kind == "ivfpq_train":
            c["n"] = min(c["n"], 300_000)
        else:
            c.update(nprobe=min(nlist, rng.choice([8, 16, 32])), rerank=rng.choice([0, 0, 100]),
                     nq=_log(rng, 1, 1024), k=rng.choice([1, 10, 10, 50]), host=rng.random() < 0.4)
        return c
    return {"kind": kind, "n": _log(rng, 20_000, 1_000_000), "dim": rng.choice([64, 96, 128, rng.randint(8, 256)]),
            "clusters": _log(rng, 16, 2048), "iterations": rng.randint(2, 10), "given": rng.random() < 0.5}


# --- inputs ---------------------------------------------------------------------------
def _centres(c):
    """Gaussian clusters, as the benchmark configurations draw them; (number, spread)."""
    if c["kind"] == "kmeans":
        return c["clusters"], 0.2
    if c["kind"] in ("ivfpq", "ivfpq_train"):
        return 1000, 0.15
    return (256, 1.0) if c["metric"] != "euclidean" else (100, 0.15)


def _inputs(c, seed):
    """(vectors [n, dim], queries [nq, dim], accept mask or None, ids to remove), from the seed alone."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    n, dim, nq = c["n"], c["dim"], c.get("nq", 0)
    if c["kind"] == "sq8":  # uniform components, as the byte-code benchmark draws them
        x = torch.rand(n, dim, generator=g, device=DEV).mul_(2.0).sub_(1.0)
        q = torch.rand(nq, dim, generator=g, device=DEV).mul_(2.0).sub_(1.0)
    else:
        clusters, sigma = _centres(c)
        centres = torch.randn(clusters, dim, generator=g, device=DEV)
        x = torch.randn(n, dim, generator=g, device=DEV).mul_(sigma)
        step = 1 << 20
        for a in range(0, n, step):
            b = min(n, a + step)
            x[a:b] += centres[torch.randint(0, clusters, (b - a,), generator=g, device=DEV)]
        q = torch.randn(nq, dim, generator=g, device=DEV).mul_(sigma)
        q += centres[torch.randint(0, clusters, (nq,), generator=g, device=DEV)]
    accept = None
    if c.get("accept", 1.0) < 1.0:
        accept = (torch.rand(n, generator=g, device=DEV) < c["accept"]).to(torch.uint8)
    removed = []
    if c.get("removed", 0):
        removed = sorted(set(torch.randint(0, n, (c["removed"],), generator=g, device=DEV).tolist()))
    return x, q, accept, removed


def _metric(c):
    return METRICS[c["metric"]]


def prepare(case, seed):
    c, kind = case, case["kind"]
    x, q, accept, removed = _inputs(c, seed)
    s = {"case": c}
    if kind == "kmeans":
        k = min(c["clusters"], c["n"])
        s.update(points=x, seed=seed, init=x[:: c["n"] // k][:k].clone() if c["given"] else None,
                 centroids=torch.zeros(k, c["dim"], device=DEV),
                 assign=torch.zeros(c["n"], dtype=torch.int32, device=DEV))
        return s
    space = px.VectorSpace(c["dim"], _metric(c))
    ids = np.arange(c["n"], dtype=np.uint64)
    if kind == "flat":
        index = px.FlatIndex(space, c["n"])
        index.insert_device(ids, x)
    elif kind == "sq8":
        index = px.Sq8Index(space, capacity=c["n"])
        sample = x[:100_000].contiguous()
        if c["metric"] == "cosine":  # ranges are fitted to prepared vectors
            sample = sample / sample.norm(dim=1, keepdim=True)
        index.train_device(sample)
        index.insert_device(ids, x)
    else:
        cfg = px.IvfPqConfig(c["nlist"], c["subspaces"]).with_train_threshold(1 << 63).with_seed(seed)
        if kind == "ivfpq":
            cfg = cfg.with_nprobe(c["nprobe"]).with_rerank(c["rerank"])
        index = px.IvfPqIndex(space, cfg)
        index.insert_device(ids, x)
        if kind == "ivfpq":
            index.train()
    for i in removed:
        index.remove(i)
    s["index"] = index
    if kind == "ivfpq_train":
        return s
    if c["host"]:
        s["queries"] = q.cpu().numpy()
    else:
        s.update(queries=q, accept=accept, ids=torch.zeros(c["nq"], c["k"], dtype=torch.int64, device=DEV),
                 dist=torch.zeros(c["nq"], c["k"], device=DEV),
                 count=torch.zeros(c["nq"], dtype=torch.int32, device=DEV))
    return s


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "kmeans":
        inertia, iterations = px.kmeans_device(s["points"], s["centroids"].shape[0], c["iterations"], s["seed"],
                                               s["centroids"], s["assign"], s["init"])
        return {"centroids": s["centroids"], "assign": s["assign"], "inertia": inertia, "iterations": iterations}
    index = s["index"]
    if c["kind"] == "ivfpq_train":
        report = index.train()
        centroids, codebooks, codes, list_of = index.parts()
        return {"centroids": centroids, "codebooks": codebooks, "codes": codes, "list_of": list_of.astype(np.int64),
                "coarse_inertia": report.coarse_inertia, "residual_inertia": report.residual_inertia}
    more = {"rescore": c["rescore"]} if c["kind"] == "sq8" else {}
    if c["host"]:
        ids, dist, count = index.search_batch(s["queries"], c["k"], **more)
        return {"ids": ids.astype(np.int64), "dist": dist, "count": count.astype(np.int64)}
    index.search_device(s["queries"], c["k"], s["ids"], s["dist"], s["count"], accept=s.get("accept"), **more)
    return {"ids": s["ids"], "dist": s["dist"], "count": s["count"]}


def work(case):
    c = case
    n, dim, nq, k = c["n"], c["dim"], c.get("nq", 0), c.get("k", 0)
    results = nq * k * 12 + nq * 4
    if c["kind"] == "flat":
        rows = n * c["accept"]
        return {"bytes": rows * dim * 4 + nq * dim * 4 + results, "flops": 2.0 * rows * dim * nq}
    if c["kind"] == "sq8":
        return {"bytes": n * dim + nq * dim * 4 + results, "flops": 2.0 * n * dim * nq}
    if c["kind"] == "ivfpq":
        lists, m, probe = c["nlist"], c["subspaces"], c["nprobe"] / c["nlist"]
        touched = n * (1.0 - (1.0 - probe) ** nq)  # entries of lists that some query probes
        return {"bytes": touched * m + lists * dim * 4 + 256 * dim * 4 + nq * dim * 4 + results,
                "flops": 2.0 * nq * lists * dim + nq * c["nprobe"] * 256 * dim * 3.0 + nq * probe * n * m}
    if c["kind"] == "ivfpq_train":
        sample, lists = min(n, 100_000), c["nlist"]
        # seeding, and at least one assignment of the sample, for both codebooks; then every vector's encoding
        once = 2.0 * dim * (lists + 256)
        return {"bytes": n * dim * 4 + n * (c["subspaces"] + 4) + (lists + 256) * dim * 4,
                "flops": 2 * sample * once + n * once}
    return {"bytes": n * dim * 4 + n * 4 + c["clusters"] * dim * 4,
            "flops": 2.0 * n * dim * c["clusters"] * (c["iterations"] + (0 if c["given"] else 1))}


def tolerance(case):
    # ids, distances, codes, centroids and sums are specified to the bit, whatever unit computes them
    return "exact"


# --- the same in 64 bits ------------------------------------------------------------------
def _unit(v):
    return v / v.norm(dim=1, keepdim=True)


def _search64(c, score, n, k, usable):
    """The k smallest scores of each query, rising; score(a, b) gives [nq, b - a] in 64 bits."""
    best = None
    step = max(1024, 120_000_000 // max(c["nq"], 1))
    for a in range(0, n, step):
        b = min(n, a + step)
        d = score(a, b)
        if usable is not None:
            d[:, ~usable[a:b]] = math.inf
        d = d.topk(min(k, b - a), largest=False, sorted=True).values
        best = d if best is None else torch.cat([best, d], 1).topk(min(k, best.shape[1] + d.shape[1]),
                                                                   largest=False, sorted=True).values
    return best


def _found(c, best):
    """Distances laid out as run() returns them: zeros past the results there are."""
    out = torch.zeros(c["nq"], c["k"], dtype=torch.float64, device=DEV)
    fine = torch.isfinite(best)
    out[:, : best.shape[1]] = torch.where(fine, best, torch.zeros_like(best))
    return {"ids": None, "dist": out.cpu().numpy(), "count": fine.sum(1).to(torch.int64).cpu().numpy()}


def exact(case, seed):
    c = case
    if c["kind"] in ("ivfpq", "ivfpq_train") or (c["kind"] == "kmeans" and not c["given"]):
        return None  # the trained centroids come from a seeded generator that plain torch does not have
    x, q, accept, removed = _inputs(c, seed)
    if c["kind"] == "kmeans":
        return _lloyd64(c, x)
    q = q.double()
    if c["kind"] == "flat":
        usable = None
        if accept is not None or removed:
            usable = torch.ones(c["n"], dtype=torch.bool, device=DEV) if accept is None else accept.bool()
            usable[torch.tensor(removed, dtype=torch.int64, device=DEV)] = False
        if c["metric"] == "cosine":
            q = _unit(q)

        def score(a, b):
            r = x[a:b].double()
            if c["metric"] == "cosine":
                return 1.0 - q @ _unit(r).T.contiguous()
            dot = q @ r.T.contiguous()
            if c["metric"] == "inner_product":
                return -dot
            return (q.square().sum(1, keepdim=True) + r.square().sum(1)[None, :] - 2.0 * dot).clamp_(min=0.0)

        return _found(c, _search64(c, score, c["n"], c["k"], usable))
    sample = x[:100_000].double()
    if c["metric"] == "cosine":
        sample, q = _unit(sample), _unit(q)
    low, scale = sample.amin(0), (sample.amax(0) - sample.amin(0)) / 255.0

    def code(v):
        return ((v - low) / scale).add_(0.5).floor_().clamp_(0.0, 255.0)

    if c["rescore"]:
        return None  # the rescored set hangs on the ties of the integer scores
    qc = code(q) - 128.0

    def score(a, b):
        r = x[a:b].double()
        return -(qc @ (code(_unit(r) if c["metric"] == "cosine" else r) - 128.0).T.contiguous())

    return _found(c, _search64(c, score, c["n"], c["k"], None))


def _lloyd64(c, x):
    n, k = c["n"], min(c["clusters"], c["n"])
    p = x.double()
    cents = p[:: n // k][:k].clone()
    norms = p.square().sum(1)
    assign = torch.full((n,), -1, dtype=torch.int64, device=DEV)
    inertia, iterations = 0.0, 0
    for it in range(c["iterations"]):
        iterations = it + 1
        new, d = torch.empty_like(assign), torch.empty(n, dtype=torch.float64, device=DEV)
        for a in range(0, n, 50_000):
            m = cents.square().sum(1)[None, :] - 2.0 * (p[a:a + 50_000] @ cents.T.contiguous())
            d[a:a + 50_000], new[a:a + 50_000] = m.min(1)
        inertia = float((d + norms).clamp(min=0.0).sum())
        if torch.equal(new, assign):
            break
        assign = new
        count = torch.bincount(assign, minlength=k)
        mean = torch.zeros_like(cents).index_add_(0, assign, p) / count.clamp(min=1)[:, None]
        part = cents  # updated in ascending order; an empty cluster takes the point farthest from it as it then is
        for e in torch.nonzero(count == 0)[:, 0].tolist():
            part = torch.cat([mean[:e], part[e:]])
            far, at = -1.0, 0
            for a in range(0, n, 50_000):
                m = part.square().sum(1)[None, :] - 2.0 * (p[a:a + 50_000] @ part.T.contiguous())
                d_far, i_far = (m.min(1).values + norms[a:a + 50_000]).max(0)
                if float(d_far) > far:
                    far, at = float(d_far), a + int(i_far)
            mean[e] = p[at]
        cents = mean
    return {"centroids": cents.cpu().numpy(), "assign": None, "inertia": inertia, "iterations": iterations}
