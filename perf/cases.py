"""Workloads of the exact k-NN framework as its users call it: sizes, inputs, one pass, and the
fp64 answer of every pass.

A case is a dict of plain values. Its "kind" names the call:

  search   Index.search over an index built beforehand, optionally stored in k-means lists
  labels   Index.search(labels=...) over a labelled (partitioned) index, the labels in GPU memory
  filter   Index.search(filter=...) with a boolean mask over the ids, or one mask per query
  decode   KeyCache.topk over a cache filled beforehand (attention, one step of decoding)
  prefill  libcertex_amd.topk: keys to a cache and its top k in one call
  graph    libcertex_amd.search(xb): the k nearest neighbours of every row, built and searched
  ingest   Index.add twice, Index.remove and Index.search on a new index

Every pass returns what the call returns: scores (or distances) and ids.
"""

import math

import torch

import libcertex_amd as certex

DEV = "cuda"
_TYPES = {"uint8": torch.uint8, "int8": torch.int8, "float32": torch.float32, "float16": torch.float16,
          "bfloat16": torch.bfloat16}
_INT = ("uint8", "int8")


def listed():
    """The workloads that are timed and compared by name."""
    return [
        # an interactive lookup: one query against a small index, bound by the calls and launches
        dict(name="lookup-u8-1q", kind="search", dtype="uint8", metric="l2", n=100_000, dim=128, nq=1, k=10,
             batch=2048, lists=0),
        # retrieval for a handful of users over a million text embeddings
        dict(name="retrieve-f32-16q", kind="search", dtype="float32", metric="cosine", n=1_000_000, dim=768, nq=16,
             k=10, batch=2048, lists=0),
        # a thousand queries against 100,000 float vectors with the default options
        dict(name="batch-f32-1kq", kind="search", dtype="float32", metric="l2", n=100_000, dim=128, nq=1000, k=10,
             batch=2048, lists=0),
        # the benchmark's workload: 10,000 queries in one batch, 10 million byte vectors in lists
        dict(name="bulk-u8-10m", kind="search", dtype="uint8", metric="l2", n=10_000_000, dim=128, nq=10_000, k=10,
             batch=10_000, lists=4096),
        # label-filtered retrieval, one tenant or category per query
        dict(name="labels-f32-10kq", kind="labels", dtype="float32", metric="cosine", n=1_000_000, dim=768,
             nq=10_000, k=100, batch=10_000, n_labels=16),
        # one mask over the ids (an access list or a date range) for all queries
        dict(name="bitset-u8-1kq", kind="filter", dtype="uint8", metric="l2", n=1_000_000, dim=128, nq=1000, k=10,
             per_query=False, keep=0.1),
        # a mask of its own for each query, half-precision embeddings
        dict(name="bitmap-f16-200q", kind="filter", dtype="float16", metric="ip", n=300_000, dim=384, nq=200, k=50,
             per_query=True, keep=0.3),
        # sparse attention over a long cache, 64 decoding sequences' queries per head
        dict(name="decode-bf16-64q", kind="decode", dtype="bfloat16", kv=8, n=131_072, dim=128, heads=32, m=64,
             k=2048),
        # the same for a single sequence: one query per head
        dict(name="decode-bf16-1q", kind="decode", dtype="bfloat16", kv=8, n=32_768, dim=128, heads=32, m=1,
             k=1024),
        # a prompt's keys and queries in one call
        dict(name="prefill-f16", kind="prefill", dtype="float16", kv=8, n=16_384, dim=64, heads=32, m=32, k=256),
        # a k-NN graph of word vectors whose dimension fits no tile
        dict(name="graph-f32-60k", kind="graph", dtype="float32", metric="cosine", n=60_000, dim=300, k=15),
        # a new index of wide byte vectors: additions, a removal, a first search
        dict(name="ingest-u8-960", kind="ingest", dtype="uint8", metric="l2", n=250_000, dim=960, nq=100, k=10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_FLOPS_MOST = 3e12  # of a drawn case (the largest listed one takes 2.6e13)


def _dim(rng):
    """A dimension in use: a round one half of the time, else any."""
    if rng.random() < 0.5:
        return rng.choice([64, 96, 128, 256, 384, 512, 768, 960, 1024])
    return _log(rng, 48, 1024)


def draw(rng):
    """One more case of the ranges of the listed ones."""
    kind = rng.choice(["search", "search", "search", "labels", "filter", "filter", "decode", "prefill", "graph",
                       "ingest"])
    if kind in ("decode", "prefill"):
        kv = rng.choice([1, 2, 4, 8])
        n = _log(rng, 2048, 131_072 if kind == "decode" else 32_768)
        return dict(kind=kind, dtype=rng.choice(["bfloat16", "float16"]), kv=kv, n=n, dim=rng.choice([64, 128]),
                    heads=kv * rng.choice([1, 4]), m=rng.choice([1, _log(rng, 2, 64)]),
                    k=min(n // 4, _log(rng, 32, 2048)))
    dtype = rng.choice(["uint8", "int8", "float32", "float32", "float16"])
    metric = rng.choice(["l2", "ip"] if dtype in _INT else ["l2", "ip", "cosine"])
    dim = _dim(rng)
    k = _log(rng, 1, 100)
    base = dict(kind=kind, dtype=dtype, metric=metric, dim=dim, k=k)
    if kind == "search":
        n = _log(rng, 10_000, 1_500_000 if dim <= 512 else 800_000)
        nq = max(1, min(_log(rng, 1, 10_000), int(_FLOPS_MOST / (2 * n * dim))))
        return dict(base, n=n, nq=nq, batch=2048, lists=rng.choice([0, 0, 0, max(16, n // 2500)]))
    if kind == "labels":
        n, labels = _log(rng, 50_000, 800_000), _log(rng, 4, 128)
        nq = max(1, min(_log(rng, 16, 10_000), int(_FLOPS_MOST * labels / (2 * n * dim))))
        return dict(base, n=n, nq=nq, batch=rng.choice([2048, 10_000]), n_labels=labels)
    if kind == "filter":
        per_query = rng.random() < 0.5
        n = _log(rng, 20_000, 300_000 if per_query else 1_000_000)
        nq = max(1, min(_log(rng, 1, 200 if per_query else 2000), int(_FLOPS_MOST / (2 * n * dim))))
        return dict(base, n=n, nq=nq, per_query=per_query, keep=rng.choice([0.05, 0.2, 0.5, 0.9]))
    if kind == "graph":
        n = min(_log(rng, 5_000, 60_000), int(math.sqrt(_FLOPS_MOST / (2 * dim))))
        return dict(base, n=n)
    return dict(base, n=_log(rng, 20_000, 250_000), nq=_log(rng, 1, 200))


# ---- inputs ------------------------------------------------------------------------------------


def _byte_rows(n, dim, g, dtype, centres):
    """Rows around shared centres, N(0, 20^2) per coordinate, rounded and clipped (image
    descriptors); int8 vectors are shifted by -64 so that both signs occur."""
    out = torch.empty((n, dim), dtype=_TYPES[dtype], device=DEV)
    step = max(1, (1 << 27) // dim)
    for i in range(0, n, step):
        m = min(step, n - i)
        c = torch.randint(0, centres.shape[0], (m,), generator=g, device=DEV)
        v = centres[c] + torch.randn((m, dim), generator=g, device=DEV) * 20.0
        if dtype == "int8":
            out[i:i + m] = (v - 64).round_().clamp_(-128, 127).to(torch.int8)
        else:
            out[i:i + m] = v.round_().clamp_(0, 255).to(torch.uint8)
    return out


def _float_rows(n, dim, g, dtype, scale, basis):
    """Embeddings: Gaussian with a power-law spectrum (variance 1 / i along the i-th direction)."""
    out = torch.empty((n, dim), dtype=_TYPES[dtype], device=DEV)
    step = max(1, (1 << 27) // dim)
    for i in range(0, n, step):
        m = min(step, n - i)
        x = (torch.randn((m, dim), generator=g, device=DEV) * scale) @ basis
        out[i:i + m] = x.to(out.dtype)
    return out


def _rows(case, seed, counts):
    """Matrices of counts[0], counts[1], ... rows of one distribution, made from the seed."""
    g = torch.Generator(device=DEV).manual_seed(1_000_003 * int(seed) + 17)
    dim = case["dim"]
    if case["dtype"] in _INT:
        centres = torch.rand((1000, dim), generator=g, device=DEV) * 80.0
        return [_byte_rows(m, dim, g, case["dtype"], centres) for m in counts]
    basis, _ = torch.linalg.qr(torch.randn((dim, dim), generator=g, device=DEV))
    scale = torch.sqrt(1.0 / torch.arange(1, dim + 1, device=DEV, dtype=torch.float32))
    return [_float_rows(m, dim, g, case["dtype"], scale, basis) for m in counts]


def _keys_and_queries(case, seed):
    """Keys N(0, 1) with 4 channels of 20 times the size (as attention keys show), queries N(0, 1)."""
    g = torch.Generator(device=DEV).manual_seed(1_000_003 * int(seed) + 41)
    t = _TYPES[case["dtype"]]
    keys = torch.randn((case["kv"], case["n"], case["dim"]), generator=g, device=DEV)
    keys[:, :, torch.randperm(case["dim"], generator=g, device=DEV)[:4]] *= 20.0
    q = torch.randn((case["heads"], case["m"], case["dim"]), generator=g, device=DEV)
    return keys.to(t), q.to(t)


def _ids_gone(case, seed):
    """Ids that the ingest case removes: about one in 64."""
    g = torch.Generator(device=DEV).manual_seed(1_000_003 * int(seed) + 43)
    return torch.randperm(case["n"], generator=g, device=DEV)[: max(1, case["n"] // 64)]


def _masks(case, seed):
    g = torch.Generator(device=DEV).manual_seed(1_000_003 * int(seed) + 47)
    shape = (case["nq"], case["n"]) if case["per_query"] else (case["n"],)
    return torch.rand(shape, generator=g, device=DEV) < case["keep"]


def _labels(case, seed):
    g = torch.Generator(device=DEV).manual_seed(1_000_003 * int(seed) + 53)
    return [torch.randint(0, case["n_labels"], (m,), generator=g, device=DEV, dtype=torch.int32)
            for m in (case["n"], case["nq"])]


def prepare(case, seed):
    """What the program holds before the call: inputs on the GPU, and the index or cache."""
    kind = case["kind"]
    state = {"case": case}
    if kind in ("decode", "prefill"):
        keys, q = _keys_and_queries(case, seed)
        state["q"] = q
        if kind == "prefill":
            state["keys"] = keys
        else:
            state["cache"] = certex.KeyCache(case["kv"], case["dim"], k=case["k"]).append(keys)
        return state
    if kind == "graph":
        (state["x"],) = _rows(case, seed, [case["n"]])
        return state
    x, state["q"] = _rows(case, seed, [case["n"], case["nq"]])
    if kind == "ingest":
        half = case["n"] - case["n"] // 3
        state["parts"] = [x[:half].contiguous(), x[half:].contiguous()]
        state["gone"] = _ids_gone(case, seed)
        return state
    index = certex.Index(case["dim"], metric=case["metric"], n_lists=case.get("lists", 0))
    if kind == "labels":
        lx, state["labels"] = _labels(case, seed)
        index.add(x, labels=lx)
    else:
        index.add(x)
    if kind == "filter":
        state["mask"] = _masks(case, seed)
    state["index"] = index
    return state


def run(state):
    """One pass."""
    case = state["case"]
    kind, k = case["kind"], case["k"]
    if kind == "search":
        # an index in lists takes its thresholds from the lists' anchors (no probe), as the benchmark does
        probe = 0 if case["lists"] and case["dtype"] in _INT else 2
        return state["index"].search(state["q"], k=k, batch=case["batch"], probe_lists=probe)
    if kind == "labels":
        return state["index"].search(state["q"], k=k, batch=case["batch"], labels=state["labels"])
    if kind == "filter":
        return state["index"].search(state["q"], k=k, filter=state["mask"])
    if kind == "decode":
        return state["cache"].topk(state["q"])
    if kind == "prefill":
        return certex.topk(state["q"], state["keys"], k)
    if kind == "graph":
        return certex.search(state["x"], k=k, metric=case["metric"])
    index = certex.Index(case["dim"], metric=case["metric"], capacity=case["n"])
    for part in state["parts"]:
        index.add(part)
    index.remove(state["gone"])
    return index.search(state["q"], k=k)


# ---- what a pass cannot do without -----------------------------------------------------------------


def work(case):
    """Every stored vector and every query read once, every result written once; two operations per
    coordinate of every (query, row) pair that the call admits."""
    size = {"uint8": 1, "int8": 1, "float32": 4, "float16": 2, "bfloat16": 2}[case["dtype"]]
    if case["kind"] in ("decode", "prefill"):
        rows, nq = case["kv"] * case["n"], case["heads"] * case["m"]
        pairs = float(nq) * case["n"]
    else:
        rows, nq = case["n"], case["n"] if case["kind"] == "graph" else case["nq"]
        pairs = float(nq) * rows
        if case["kind"] == "labels":
            pairs /= case["n_labels"]
        if case["kind"] == "filter":
            pairs *= case["keep"]
    given = 0
    if case["kind"] == "filter":
        given = case["n"] * (nq if case["per_query"] else 1)
    elif case["kind"] == "labels":
        given = 4 * nq
    return {"bytes": float((rows + (0 if case["kind"] == "graph" else nq)) * case["dim"] * size + nq * case["k"] * 12
                           + given),
            "flops": 2.0 * pairs * case["dim"]}


def tolerance(case):
    """Byte vectors: every score is a whole number, and equal scores go to the lower id. Float
    vectors: scores are fp64 sums returned as float32 (cosine similarities as 1 - float32(1 - c))."""
    if case["dtype"] in _INT:
        return "exact"
    return {"rel": 2e-7, "max": 5e-7, "differ": 1e-5}


# ---- the answer in 64 bits ---------------------------------------------------------------------------


def _best(scores, k, integer):
    """The k smallest scores of every row and their columns, equal scores by the lower column."""
    if integer:
        key = scores.long() * (1 << 31) + torch.arange(scores.shape[1], device=scores.device)
        key = key.topk(k, dim=1, largest=False).values.sort(1).values
        return (key >> 31).double(), key & ((1 << 31) - 1)
    v, i = scores.topk(k, dim=1, largest=False)
    order = v.argsort(dim=1, stable=True)
    return v.gather(1, order), i.gather(1, order)


def _knn64(X, Q, k, metric, integer, keep=None):
    """Scores (smaller is better) and ids of the k best rows of X for every query, in fp64; `keep`
    (queries, rows) -> the admitted pairs, called with a range of queries."""
    Xd = X.double()
    if metric == "cosine":
        Xd = Xd / Xd.norm(dim=1, keepdim=True)
    xx = Xd.square().sum(1)
    step = max(1, (1 << 28) // X.shape[0])
    vs, ids = [], []
    for i in range(0, Q.shape[0], step):
        q = Q[i:i + step].double()
        if metric == "cosine":
            q = q / q.norm(dim=1, keepdim=True)
        s = -(q @ Xd.T)
        if metric == "l2":
            s = q.square().sum(1, keepdim=True) + 2 * s + xx
        lowest = float(1 << 31) if integer else math.inf
        if keep is not None:
            s = s.masked_fill(~keep(i, i + q.shape[0]), lowest)
        v, j = _best(s, k, integer)
        if metric == "l2" and not integer:  # the sum over the differences has no cancellation
            order_rows = Xd[j.reshape(-1)].reshape(j.shape[0], k, -1)
            w = (q[:, None, :] - order_rows).square().sum(-1).masked_fill(torch.isinf(v), math.inf)
            order = w.argsort(dim=1, stable=True)
            v, j = w.gather(1, order), j.gather(1, order)
        j = j.masked_fill(v == lowest, -1)
        vs.append(v.masked_fill(v == lowest, math.inf))
        ids.append(j)
    v, j = torch.cat(vs), torch.cat(ids)
    return (v if metric == "l2" else -v), j


def exact(case, seed):
    """What run() returns, in fp64; None where that takes too long."""
    if case["n"] * float(case.get("nq", case["n"])) * (case.get("n_labels", 1) ** -1) > 2e10:
        return None
    k, integer = case["k"], case["dtype"] in _INT
    if case["kind"] in ("decode", "prefill"):
        keys, q = _keys_and_queries(case, seed)
        r = case["heads"] // case["kv"]
        out = [_knn64(keys[h // r], q[h], k, "ip", False) for h in range(case["heads"])]
        return torch.stack([v for v, _ in out]), torch.stack([j for _, j in out])
    if case["kind"] == "graph":
        (x,) = _rows(case, seed, [case["n"]])
        return _knn64(x, x, k, case["metric"], integer)
    x, q = _rows(case, seed, [case["n"], case["nq"]])
    keep = None
    if case["kind"] == "ingest":
        alive = torch.ones(case["n"], dtype=torch.bool, device=DEV)
        alive[_ids_gone(case, seed)] = False
        keep = lambda a, b: alive.expand(b - a, -1)  # noqa: E731
    elif case["kind"] == "filter":
        mask = _masks(case, seed)
        keep = (lambda a, b: mask[a:b]) if case["per_query"] else (lambda a, b: mask.expand(b - a, -1))
    elif case["kind"] == "labels":
        lx, lq = _labels(case, seed)
        v = torch.empty((case["nq"], k), dtype=torch.float64, device=DEV)
        j = torch.empty((case["nq"], k), dtype=torch.int64, device=DEV)
        for label in lq.unique().tolist():
            rows, at = (lx == label).nonzero()[:, 0], (lq == label).nonzero()[:, 0]
            kk = min(k, rows.shape[0])
            v[at], j[at] = (math.inf if case["metric"] == "l2" else -math.inf), -1
            if kk > 0:
                vv, jj = _knn64(x[rows], q[at], kk, case["metric"], integer)
                v[at, :kk], j[at, :kk] = vv, rows[jj]
        return v, j
    return _knn64(x, q, k, case["metric"], integer, keep)
