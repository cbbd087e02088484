"""The work whose speed is followed: searches, streamed searches and index
builds through the package's public entry points, over the sizes that users of
this library run.

A case is a dict of plain values.  Its "kind" says what one pass is:

- "request": a query batch straight from host arrays through
  search_noalloc, the one-call serving path.
- "fresh": a query batch that did not exist before: Index.batch, stages A and
  B, the search, Batch.close.
- "search": stages A and B and the search on a batch that the program keeps
  (the driver's sweep over L, a serving loop over resident queries).
- "stream": the arithmetic-grid stage A and the search of a streamed
  (out-of-core) index.
- "build": the index build from host arrays: grid, exact kNN graphs,
  their optimisation, cross edges, k-means labels.

Results are exact by contract: the library sums distances in one fixed order
and breaks ties by row, so every kind is compared bit for bit.
"""
import math

import numpy as np
import torch

import garfield_amd as gf

DOMAIN = 10000   # attribute values are integers in [0, DOMAIN)
ROWS = {"f32": gf.VEC_F32, "f16": gf.VEC_F16, "u8": gf.VEC_U8, "i8q": gf.VEC_I8Q, "f16ref": gf.VEC_F16_REF}


def _search(**kw):
    """A case of kind request, fresh or search: defaults of the reference's
    driver (K = 10, recycle list 10, top 4 centres, no postfilter)."""
    c = dict(data="int", rows="f32", attrs="uniform", a=2, grid="4x4", R=32, E=2, C=100, sel_lo=0.01, sel_hi=0.5,
             prefilter=0.05, L=100, K=10, channels=1, postfilter=0)
    c.update(kw)
    return c


def listed():
    return [
        # One query of an interactive program, host arrays in and out: the
        # smallest call there is.
        _search(name="request_one", kind="request", N=100_000, D=128, R=16, Q=1, prefilter=0.05, L=64),
        # A few dozen users' queries collected by a server, most of them
        # narrow enough for the filtered brute force (prefilter 0.3).
        _search(name="request_small", kind="request", N=100_000, D=128, R=16, Q=48, prefilter=0.3, L=64),
        # A thousand new queries on a small index, batch object and all
        # (the 100k x 128 configuration).
        _search(name="fresh_1k", kind="fresh", N=100_000, D=128, R=16, Q=1000, sel_lo=0.3, sel_hi=0.3,
                prefilter=0.1, L=64),
        # The headline configuration: 1M x 128 integers, 10k queries, every
        # query exact.
        _search(name="exact_int_1m", kind="search", N=1_000_000, D=128, C=1000, Q=10_000, prefilter=1.0, L=10),
        # Cell-by-cell traversal of every query, fp32 rows.
        _search(name="traverse_f32", kind="search", N=250_000, D=128, C=500, Q=2500, prefilter=0.0, L=100),
        # Binary16 rows (the driver's default), skewed attributes on 64 cells,
        # a long list.
        _search(name="traverse_f16", kind="search", data="unit", rows="f16", attrs="zipf", a=3, grid="4x4x4",
                N=200_000, D=96, C=300, Q=1200, sel_lo=0.001, prefilter=0.05, L=250),
        # The dual-channel traversal at a recall-oriented list length, u8
        # rows, beside the brute force for the narrow queries.
        _search(name="dual_u8", kind="search", rows="u8", N=250_000, D=128, C=500, Q=2500, prefilter=0.2, L=600,
                channels=2),
        # Float rows, every query exact: 96-d unit vectors with skewed
        # attributes, fp32.
        _search(name="exact_f32", kind="search", data="unit", attrs="zipf", a=3, grid="4x4x4", N=300_000, D=96,
                C=300, Q=3001, sel_lo=0.001, prefilter=1.0, L=10),
        # 768-d embeddings stored in binary16, attributes tied to their topic.
        _search(name="exact_f16_768", kind="search", data="mixture", rows="f16", N=120_000, D=768, C=200, Q=4096,
                sel_lo=0.1, sel_hi=0.1, prefilter=1.0, L=10),
        # Odd sizes: 100-d vectors, a point count and a query count that
        # nothing divides.
        _search(name="exact_ragged", kind="search", data="unit", N=150_001, D=100, C=150, Q=777, prefilter=1.0, L=10),
        # Out of core: u8 rows on a 16 x 16 arithmetic grid, 16 cells a batch.
        dict(name="stream_u8", kind="stream", N=150_000, D=128, R=32, E=2, grid="16x16", Q=4000, sel_lo=0.005,
             sel_hi=0.2, threshold=1.0, L=32, K=10),
        # The index of 200k integer vectors from nothing.
        dict(name="build_int", kind="build", data="int", N=200_000, D=128, a=2, grid="4x4", R=32, inter=64, E=2,
             C=200, iters=8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["request", "fresh", "search", "search", "search", "search", "stream", "build"])
    if kind == "stream":
        sel = _log_int(rng, 20, 400) / 1000.0
        return dict(kind="stream", N=_log_int(rng, 30_000, 150_000), D=rng.choice([64, 96, 112, 128, 256]), R=rng.choice([16, 32]),
                    E=rng.choice([1, 2]), grid=rng.choice(["8x8", "16x16"]), Q=_log_int(rng, 50, 4000), sel_lo=sel / 20,
                    sel_hi=sel, threshold=rng.choice([1.0, 1.0, 0.25]), L=rng.choice([32, 64, 100]), K=10)
    if kind == "build":
        data = rng.choice(["int", "int", "unit"])
        return dict(kind="build", data=data, N=_log_int(rng, 10_000, 180_000), D=rng.choice([64, 96, 100, 128, 200]), a=2,
                    grid=rng.choice(["4x4", "2x4", "3x3"]), R=rng.choice([16, 24, 32]),
                    inter=64 if data == "int" else 47, E=rng.choice([1, 2]), C=_log_int(rng, 20, 300), iters=rng.choice([4, 8]))
    data, rows = rng.choice([("int", "f32"), ("int", "u8"), ("unit", "f32"), ("unit", "f16"), ("unit", "i8q"),
                             ("mixture", "f16"), ("unit", "f16ref")])
    if kind == "request" and rows == "i8q":
        rows = "f32"
    D = rng.choice({"f32": [64, 96, 100, 128, 200, 256], "f16": [64, 96, 104, 128, 200, 256, 384, 768],
                    "f16ref": [96, 128, 256], "u8": [64, 96, 128, 208], "i8q": [96, 128, 208]}[rows])
    a = rng.choice([1, 2, 2, 3])
    zipf = data == "unit" and a == 3
    c = _search(kind=kind, data=data, rows=rows, attrs="zipf" if zipf else "uniform", a=a,
                grid={1: "8", 2: rng.choice(["4x4", "2x5"]), 3: rng.choice(["2x2x2", "4x4x4"])}[a],
                N=_log_int(rng, 15_000, 250_000 if D <= 256 else 100_000), D=D, R=rng.choice([16, 32]),
                E=rng.choice([1, 2]), C=_log_int(rng, 16, 500), sel_lo=rng.choice([0.001, 0.01, 0.1]), sel_hi=0.5,
                prefilter=rng.choice([0.0, 0.05, 0.3, 1.0, 1.0]), L=rng.choice([10, 32, 64, 100, 250, 500]),
                K=rng.choice([5, 10, 10, 20]))
    c["Q"] = {"request": lambda: _log_int(rng, 1, 64), "fresh": lambda: _log_int(rng, 8, 2000),
              "search": lambda: _log_int(rng, 40, 4000)}[kind]()
    if kind == "search" and c["R"] <= 32:
        c["channels"] = rng.choice([1, 1, 2])
        c["postfilter"] = rng.choice([0, 0, 0, 8])
    if c["L"] > 250 and c["prefilter"] < 0.3:
        c["Q"] = min(c["Q"], 1000)
    c["L"] = max(c["L"], c["K"])
    return c


# --------------------------------------------------------------- inputs
def _grid(case):
    return [int(x) for x in case["grid"].split("x")]


def _vectors(case, n, gen, centres=None):
    """n vectors and, for a mixture, their components, as host arrays."""
    D, dev = case["D"], "cuda"
    if case["data"] == "int":
        return torch.randint(0, 256, (n, D), generator=gen, device=dev, dtype=torch.uint8).float().cpu().numpy(), None
    if case["data"] == "unit":
        x = torch.randn((n, D), generator=gen, device=dev)
        return (x / x.norm(dim=1, keepdim=True)).cpu().numpy(), None
    comp = torch.randint(0, centres.shape[0], (n,), generator=gen, device=dev)
    x = centres[comp] + 0.1 * torch.randn((n, D), generator=gen, device=dev)
    return x.cpu().numpy(), comp.cpu().numpy()


def _points(case, seed):
    """The indexed points: vectors and integer attributes; the mixture's
    centres and the generator go on to the queries."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 7919 + 17)
    rng = np.random.default_rng(int(seed) * 104729 + 5)
    N, a = case["N"], case.get("a", 2)
    centres = None
    if case["data"] == "mixture":
        centres = torch.randn((1000, case["D"]), generator=gen, device="cuda")
        centres /= centres.norm(dim=1, keepdim=True)
    vec, comp = _vectors(case, N, gen, centres)
    if case["data"] == "mixture":     # attributes follow the topic
        att = 10 * comp[:, None] + rng.integers(0, 10, size=(N, a))
    elif case.get("attrs") == "zipf":
        att = np.minimum(rng.zipf(1.1, size=(N, a)) - 1, DOMAIN - 1)
    else:
        att = rng.integers(0, DOMAIN, size=(N, a))
    return vec, att.astype(np.int32), gen, rng, centres


def _queries(case, att, gen, rng, centres):
    """Query vectors and closed ranges, selectivity log-uniform in
    [sel_lo, sel_hi]: each range holds sel**(1/a) of the points' values on
    every attribute."""
    Q, N, a = case["Q"], case["N"], att.shape[1]
    q, _ = _vectors(case, Q, gen, centres)
    sel = np.exp(rng.uniform(math.log(case["sel_lo"]), math.log(case["sel_hi"]), size=Q))
    w = np.clip(np.round(N * sel ** (1.0 / a)), 1, N).astype(np.int64)
    lo = np.empty((Q, a), np.float32)
    hi = np.empty((Q, a), np.float32)
    for d in range(a):
        s = np.sort(att[:, d])
        r0 = (rng.random(Q) * (N - w + 1)).astype(np.int64)
        lo[:, d] = s[r0]
        hi[:, d] = s[r0 + w - 1]
    return q, lo, hi


def _stream_case(case):
    return dict(case, data="int", a=2)


def _arith_width(case):
    return [float((DOMAIN + g - 1) // g) for g in _grid(case)]


# --------------------------------------------------------------- prepare
def _quantiles(l_q, r_q):
    return np.concatenate(l_q).astype(np.float32), np.concatenate(r_q).astype(np.float32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "build":
        vec, att, _, rng, _ = _points(case, seed)
        if case["data"] == "int":
            vec = vec.astype(np.uint8)
        init = rng.choice(case["N"], size=case["C"], replace=False).astype(np.uint32)
        return dict(case=case, vec=vec, att=att.astype(np.float32), init=init)
    if kind == "stream":
        c = _stream_case(case)
        vec, att, gen, rng, _ = _points(c, seed)
        grid, width = _grid(c), _arith_width(c)
        P = int(np.prod(grid))
        idx = [np.minimum(att[:, d] // int(width[d]), grid[d] - 1) for d in range(2)]
        pid = (idx[0] * grid[1] + idx[1]).astype(np.uint32)
        l_q = [np.array([j * width[d] for j in range(grid[d])]) for d in range(2)]
        r_q = [np.array([(j + 1) * width[d] - 1 for j in range(grid[d])]) for d in range(2)]
        graphs, cross, _ = gf.build_graphs(vec.astype(np.uint8), pid, P, c["R"], c["E"])
        lq, rq = _quantiles(l_q, r_q)
        ix = gf.Index.create_streamed(vec, att.astype(np.float32), grid, lq, rq, pid, graphs, cross, batch_cells=16,
                                      vec_dtype=gf.VEC_U8)
        q, lo, hi = _queries(c, att, gen, rng, None)
        return dict(case=case, ix=ix, batch=ix.batch(q, lo, hi), amin=np.zeros(2, np.float32),
                    width=np.array(width, np.float32), out=_out(case))
    vec, att, gen, rng, centres = _points(case, seed)
    grid = _grid(case)
    P = int(np.prod(grid))
    lq, rq, _, pid = gf.grid_scatter(att.astype(np.float32), grid)
    v = vec.astype(np.uint8) if case["data"] == "int" else vec
    graphs, cross, _ = gf.build_graphs(v, pid, P, case["R"], case["E"])
    labels, _, _ = gf.kmeans(v, case["C"], 2, seed=int(seed) % 1000)
    lq, rq = _quantiles(lq, rq)
    ix = gf.Index.from_arrays(vec, att.astype(np.float32), grid, lq, rq, pid, graphs, cross, labels=labels,
                              vec_dtype=ROWS[case["rows"]])
    q, lo, hi = _queries(case, att, gen, rng, centres)
    s = dict(case=case, ix=ix, q=q, lo=lo, hi=hi, out=_out(case))
    if case["kind"] == "search":
        s["batch"] = ix.batch(q, lo, hi)
    return s


def _out(case):
    """The page-locked result arrays that a program which searches in a loop
    keeps."""
    shape = (case["Q"], case["K"])
    return gf.pinned_empty(shape, np.uint32), gf.pinned_empty(shape, np.float32)


# --------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "build":
        lq, rq, _, pid = gf.grid_scatter(state["att"], _grid(case))
        P = int(np.prod(_grid(case)))
        knn, cross, _ = gf.build_graphs(state["vec"], pid, P, case["inter"], case["E"])
        sizes = np.bincount(pid, minlength=P)
        graphs, _ = gf.optimize_graphs(knn, sizes, case["R"])
        labels, centres, _ = gf.kmeans(state["vec"], case["C"], case["iters"], init_ids=state["init"])
        return dict(l_q=np.concatenate(lq), r_q=np.concatenate(rq), pid=pid, knn=knn, cross=cross, graphs=graphs,
                    labels=labels, centres=centres)
    if kind == "stream":
        b = state["batch"]
        b.mark_cells_grid(state["amin"], state["width"], case["threshold"])
        ids, dists, _ = b.search(L=case["L"], K=case["K"], out=state["out"])
        return dict(ids=ids, dists=dists)
    post = case["postfilter"] or 1 << 30
    if kind == "request":
        ids, dists = gf.search_noalloc(state["ix"], state["q"], state["lo"], state["hi"], case["prefilter"], topc=4,
                                       L=case["L"], K=case["K"], postfilter=post, out=state["out"])
        return dict(ids=ids, dists=dists)
    b = state["batch"] if kind == "search" else state["ix"].batch(state["q"], state["lo"], state["hi"])
    b.mark_cells(case["prefilter"], timed=False)
    b.order_cells(4, timed=False)
    ids, dists, _ = b.search(L=case["L"], K=case["K"], postfilter=post, out=state["out"], channels=case["channels"])
    if kind == "fresh":
        b.close()
    return dict(ids=ids, dists=dists)


# --------------------------------------------------------- work, tolerance
def _mean_sel(lo, hi):
    return lo if hi <= lo else (hi - lo) / math.log(hi / lo)


def work(case):
    """Bytes: points, attributes, queries and results once.  Operations: two
    per dimension of each (query, passing point) pair of an exact search, of
    each row that a traversal has to evaluate (its list's L entries in each
    cell that a range reaches, at least), of each pair of an exact build."""
    N, D, kind = case["N"], case["D"], case["kind"]
    if kind == "build":
        P = int(np.prod(_grid(case)))
        row = 1 if case["data"] == "int" else 4
        pairs = N * N / P + N * N + (case["iters"] + 1) * N * case["C"]
        return {"bytes": N * (D * row + 8 + 4 * (1 + case["inter"] + P * case["E"] + case["R"] + 1)), "flops": 2.0 * D * pairs}
    Q, K = case["Q"], case["K"]
    sel = _mean_sel(case["sel_lo"], case["sel_hi"])
    rows = case.get("rows", "u8")
    rb = D * {"f32": 4, "f16": 2, "f16ref": 2, "u8": 1, "i8q": 1}[rows]
    a = case.get("a", 2)
    lo, hi = case["sel_lo"], case["sel_hi"]
    pf = case["threshold"] if kind == "stream" else case["prefilter"]
    if pf >= 1.0 or kind == "stream":
        exact = 1.0
    elif pf <= lo:
        exact = 0.0
    elif pf >= hi:
        exact = 1.0
    else:
        exact = math.log(pf / lo) / math.log(hi / lo)
    passing = Q * exact * N * (sel if exact == 1.0 else _mean_sel(lo, min(hi, pf)) if exact else 0.0)
    P = int(np.prod(_grid(case)))
    reach = max(1.0, P * sel)
    walked = Q * (1.0 - exact) * reach * case["L"]
    touched = min(float(N), passing + walked)
    return {"bytes": touched * (rb + 4 * a) + walked * 4 * case["R"] + Q * (4 * D + 8 * a + 8 * K),
            "flops": 2.0 * D * (passing + walked)}


def tolerance(case):
    """Ids, distances (one fixed summation order, ties by row) and builds
    (integer distances) have one right answer, bit for bit."""
    return "exact"


# ----------------------------------------------------------------- exact
def exact(case, seed):
    """Distances of the exact filtered search in 64 bits, over the rows as
    stored (binary16 rows: of the rounded values).  None for ids (ties),
    for traversals, for arithmetic that is the reference's own (f16ref,
    i8q) and for builds, which hold integers only."""
    kind = case["kind"]
    if kind == "build" or case.get("rows") in ("f16ref", "i8q"):
        return None
    c = _stream_case(case) if kind == "stream" else case
    if (c["threshold"] if kind == "stream" else c["prefilter"]) < 1.0:
        return None
    if kind != "stream" and c["postfilter"]:
        return None
    vec, att, gen, rng, centres = _points(c, seed)
    q, lo, hi = _queries(c, att, gen, rng, centres)
    x = torch.from_numpy(vec).cuda()
    y = torch.from_numpy(q).cuda()
    if c.get("rows") == "f16":
        x, y = x.half(), y.half()
    x, y = x.double(), y.double()
    at = torch.from_numpy(att).cuda().float()
    l, h = torch.from_numpy(lo).cuda(), torch.from_numpy(hi).cuda()
    xn = (x * x).sum(1)
    K = c["K"]
    res = torch.empty((len(q), K), dtype=torch.float64, device="cuda")
    for s in range(0, len(q), 256):
        e = min(len(q), s + 256)
        yy = y[s:e]
        d = (yy * yy).sum(1, keepdim=True) + xn[None, :] - 2.0 * (yy @ x.T)
        ok = torch.ones_like(d, dtype=torch.bool)
        for j in range(at.shape[1]):
            ok &= (at[None, :, j] >= l[s:e, None, j]) & (at[None, :, j] <= h[s:e, None, j])
        d = torch.where(ok, d.clamp_min(0.0), torch.full_like(d, float("inf")))
        i = torch.topk(d, K, dim=1, largest=False).indices
        # the K rows' distances again as a sum of squares, free of the
        # product form's cancellation
        v = ((x[i] - yy[:, None, :]) ** 2).sum(2)
        res[s:e] = torch.where(torch.isfinite(d.gather(1, i)), v, torch.full_like(v, float("inf"))).sort(dim=1).values
    return dict(ids=None, dists=res.cpu().numpy())
