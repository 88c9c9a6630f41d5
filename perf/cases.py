"""The SCC work this package is used for, as cases a timing program can run.

A case is a dict of plain values.  prepare(case, seed) makes what a caller
has in hand before the call (a context with its resident graph, a batch, a
running server, or host arrays, and the buffer its labels go to), run(state)
is one pass through the public entry points, and its outputs are the
canonical labels (each vertex's smallest fellow member) with the SCC counts.

Callers of the C interface own the label buffer and keep it from call to
call, so the resident cases read their labels with scc_labels or
scc_batch_labels into one page-locked buffer; the one-shot and serving cases
go through the Python host interface, which returns new arrays.
"""
import ctypes
import math

import numpy as np
import torch

import detectingscc_amd as scc

_u32p = ctypes.POINTER(ctypes.c_uint32)


def listed():
    return [
        # the smallest calls: a graph of the sample files' size, where launches
        # and looks at the counters are the whole time; an odd vertex count
        dict(name="er-999", kind="er", V=999, draws=4001, cycles=4, cmax=32, algo="g", trim1=True, trim2=True),
        # one small Erdos-Renyi graph with planted cycles, all phases on
        dict(name="er-16k", kind="er", V=16384, draws=131072, cycles=64, cmax=256, algo="g", trim1=True,
             trim2=True),
        # a host graph solved once: upload, decomposition, labels (what the
        # drop-in drivers do on every call)
        dict(name="rmat-18-solve", kind="solve", scale=18, E=16 << 18, algo="g", trim1=True, trim2=True),
        # a resident graph with sizes: labels, largest SCC and the size
        # histogram; an arc count that is no multiple of anything
        dict(name="rmat-20-sizes", kind="rmat", scale=20, E=(16 << 20) - 77, algo="g", trim1=True, trim2=True,
             sizes=True),
        # the power-law graph of the algorithm matrix, Hong's order
        dict(name="rmat-22", kind="rmat", scale=22, E=16 << 22, algo="g", trim1=True, trim2=True, sizes=False),
        # the same by colouring with the trims off: the colour rounds and the
        # multi-class searches carry the millions of trivial SCCs
        dict(name="rmat-22-colour", kind="rmat", scale=22, E=16 << 22, algo="h", trim1=False, trim2=False,
             sizes=False),
        # the large power-law graph
        dict(name="rmat-24", kind="rmat", scale=24, E=16 << 24, algo="g", trim1=True, trim2=True, sizes=False),
        # the high-diameter graph: thousands of narrow levels
        dict(name="grid-4096", kind="grid", side=4096, p=0.7, algo="g", trim1=True, trim2=True),
        # partitioned: local SCCs of 200 communities, then the merge
        dict(name="parts-8m", kind="parts", V=1 << 23, K=200, deg=12.0, inter=0.02),
        # thousands of graphs of very different sizes in one persistent launch
        dict(name="batch-4096", kind="batch", graphs=4096, lgmin=8, lgmax=16, lanes=16, block=1024),
        # a batch of small graphs with the default launch options
        dict(name="batch-small", kind="batch", graphs=700, lgmin=8, lgmax=12, lanes=4, block=256),
        # requests of mixed sizes arriving together at the server
        dict(name="serve-48", kind="serve", requests=48, median=16384, sigma=1.5, vcap=1 << 20, degree=8.0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["er", "er", "solve", "rmat", "rmat", "rmat", "grid", "parts", "batch", "serve"])
    trims = rng.random() < 0.8
    if kind == "er":
        V = _log_int(rng, 200, 200_000)
        return dict(kind=kind, V=V, draws=int(V * rng.uniform(2.0, 9.0)), cycles=rng.randint(0, 64), cmax=32,
                    algo=rng.choice("gghx"), trim1=trims, trim2=trims)
    if kind == "solve":
        s = rng.randint(12, 19)
        return dict(kind=kind, scale=s, E=int((1 << s) * rng.uniform(4, 16)), algo=rng.choice("gx"), trim1=True,
                    trim2=True)
    if kind == "rmat":
        s = rng.randint(14, 23)
        algo = rng.choice("ggghy")
        return dict(kind=kind, scale=s, E=int((1 << s) * rng.uniform(6, 16)) | 1, algo=algo, trim1=trims,
                    trim2=trims, sizes=rng.random() < 0.3)
    if kind == "grid":
        return dict(kind=kind, side=_log_int(rng, 48, 3000), p=round(rng.uniform(0.62, 0.85), 3), algo="g",
                    trim1=True, trim2=True)
    if kind == "parts":
        return dict(kind=kind, V=_log_int(rng, 1 << 16, 1 << 23), K=rng.randint(20, 300),
                    deg=round(rng.uniform(8.0, 12.0), 2), inter=0.02)
    if kind == "batch":
        lo = rng.randint(6, 10)
        block = rng.choice([256, 512, 1024])
        return dict(kind=kind, graphs=_log_int(rng, 64, 2048), lgmin=lo, lgmax=rng.randint(lo + 1, 16),
                    lanes=rng.choice([4, 16]), block=block)
    return dict(kind=kind, requests=rng.randint(8, 48), median=_log_int(rng, 2048, 16384), sigma=1.2,
                vcap=1 << 20, degree=round(rng.uniform(4.0, 10.0), 2))


# ------------------------------------------------------------- inputs ---

def _er_arcs(case, seed):
    """Uniform arcs without self-loops plus directed cycles over random
    vertices: the arcs sorted by (source, target), 1-based."""
    rng = np.random.default_rng([seed, case["V"], case["draws"]])
    V = case["V"]
    src = rng.integers(1, V + 1, size=case["draws"])
    dst = rng.integers(1, V + 1, size=case["draws"])
    keep = src != dst
    parts = [np.stack([src[keep], dst[keep]])]
    for _ in range(case["cycles"]):
        ring = rng.permutation(V)[:int(rng.integers(2, min(case["cmax"], V) + 1))] + 1
        parts.append(np.stack([ring, np.roll(ring, -1)]))
    arcs = np.concatenate(parts, axis=1).astype(np.int64)
    key = np.sort(arcs[0] * (V + 1) + arcs[1])
    return key // (V + 1), key % (V + 1)


def _csr(V, src, dst):
    """Reference layout: rows of V+2 offsets (vertex 0 empty) and columns."""
    rows = np.zeros(V + 2, np.int64)
    np.cumsum(np.bincount(src, minlength=V + 1)[:V + 1], out=rows[1:])
    return rows.astype(np.uint32), dst.astype(np.uint32)


def _er_graph(case, seed):
    V = case["V"]
    src, dst = _er_arcs(case, seed)
    Fr, Fc = _csr(V, src, dst)
    back = np.argsort(dst, kind="stable")
    Br, Bc = _csr(V, dst[back], src[back])
    return scc.Graph(V, int(src.size), Fr, Fc, Br, Bc)


def _request_sizes(case):
    """Vertices of each request: lognormal, the same for every seed (the
    requests' arcs are what the seed draws)."""
    rng = np.random.default_rng(case["requests"])
    V = case["median"] * np.exp(case["sigma"] * rng.standard_normal(case["requests"]))
    return [int(v) for v in np.clip(V, 2, case["vcap"])]


def _buffer(words):
    return torch.zeros(words, dtype=torch.int32, pin_memory=True)


def prepare(case, seed):
    kind = case["kind"]
    ctx = scc.Context(0)
    st = {"case": case, "kind": kind, "ctx": ctx}
    if kind == "solve":
        # host arrays, as a program that has loaded a graph file holds them
        st["graph"] = scc.gen_rmat(case["scale"], E=case["E"], seed=1 + seed)
        return st
    if kind == "serve":
        st["graphs"] = [scc.gen_serving_mix(1, V, 0.0, case["vcap"], case["degree"], seed=1 + seed * 64 + i).graph(0)
                        for i, V in enumerate(_request_sizes(case))]
        ctx.server_start(budget_bytes=16 << 30, max_batch=256, slots=3, solo_vertices=1 << 16, lanes=16, block=1024)
        return st
    if kind == "batch":
        ctx.gen_batch_mix_dev(case["graphs"], case["lgmin"], case["lgmax"], 2.0, 16.0, seed=1 + seed)
        # the label buffer of a program that runs batch after batch of such a
        # mix: the mean number of rows and six standard deviations more
        n, lo, hi = case["graphs"], 1 << case["lgmin"], 1 << case["lgmax"]
        words = int(n * (2 + (hi - lo) / math.log(hi / lo)) + 2 * hi * math.sqrt(n))
        if int(ctx.batch_info().row_off[-1]) > words:
            raise RuntimeError("the batch does not fit its label buffer")
        st["labels"] = _buffer(words)
        st["counts"] = torch.zeros(n, dtype=torch.int32)
        return st
    if kind == "er":
        ctx.upload(_er_graph(case, seed))
    elif kind == "rmat":
        ctx.gen_rmat_dev(case["scale"], E=case["E"], seed=1 + seed)
    elif kind == "grid":
        ctx.gen_grid_dev(case["side"], case["p"], seed=1 + seed)
    elif kind == "parts":
        ctx.gen_communities_dev(case["V"], case["K"], case["deg"], case["inter"], seed=1 + seed)
    st["labels"] = _buffer(ctx.graph.V + 1)
    return st


def _ptr(t):
    return ctypes.cast(t.data_ptr(), _u32p)


def run(st):
    case, ctx, kind = st["case"], st["ctx"], st["kind"]
    if kind == "solve":
        lab, stats = ctx.solve(st["graph"], algo=case["algo"], trim1=case["trim1"], trim2=case["trim2"],
                               sizes=False)
        return {"labels": lab, "sccs": stats.num_sccs}
    if kind == "serve":
        ids = [ctx.server_submit(g) for g in st["graphs"]]
        ctx.server_wait_all()
        return [ctx.server_poll(i)[0] for i in ids]
    if kind == "batch":
        ctx.batch_run(lanes=case["lanes"], block=case["block"])
        if scc.lib().scc_batch_labels(ctx._ctx, _ptr(st["labels"]), _ptr(st["counts"])) != 0:
            raise RuntimeError("scc_batch_labels failed")
        return {"labels": st["labels"], "sccs": st["counts"]}
    sizes = bool(case.get("sizes", False))
    algo = "d" if kind == "parts" else case["algo"]
    stats = ctx.run(algo=algo, trim1=case.get("trim1", True), trim2=case.get("trim2", True), sizes=sizes)
    if scc.lib().scc_labels(ctx._ctx, _ptr(st["labels"])) != 0:
        raise RuntimeError("scc_labels failed")
    out = {"labels": st["labels"], "sccs": stats.num_sccs}
    if sizes:
        out["largest"] = stats.largest
        out["histogram"] = np.array(ctx.histogram()[0], np.int64)
    return out


# --------------------------------------------------------- work, exact ---

def _sizes_of(case):
    """Vertices and arcs, expected ones where the inputs are drawn."""
    kind = case["kind"]
    if kind == "er":
        return case["V"], case["draws"] + case["cycles"] * case["cmax"] // 2
    if kind in ("solve", "rmat"):
        return 1 << case["scale"], case["E"]
    if kind == "grid":
        n = case["side"]
        return n * n, int(4 * n * (n - 1) * case["p"])
    if kind == "parts":
        return case["V"], int(case["V"] * case["deg"])
    if kind == "batch":   # V log-uniform in [2^lgmin, 2^lgmax], degree uniform in [2, 16]
        lo, hi = 1 << case["lgmin"], 1 << case["lgmax"]
        V = int(case["graphs"] * (hi - lo) / math.log(hi / lo))
        return V, 9 * V
    V = sum(_request_sizes(case))
    return V, int(V * case["degree"])


def work(case):
    """Bytes: every arc seen once from its source (row offsets and columns of
    the forward CSR) and every label written; a one-shot call or a request
    also brings the whole host graph, both CSRs, to the device.  No floating
    point work."""
    V, E = _sizes_of(case)
    csr = 4 * (V + 2) + 4 * E
    if case["kind"] in ("solve", "serve"):
        csr *= 2
    return {"bytes": csr + 4 * (V + 1), "flops": 0}


def exact(case, seed):
    """Tarjan's algorithm on the same arcs, for the graphs made here; the
    other outputs are whole numbers of generated graphs too large for it."""
    if case["kind"] != "er" or case["V"] + case["draws"] > 2_000_000:
        return None
    V = case["V"]
    src, dst = _er_arcs(case, seed)
    Fr, Fc = _csr(V, src, dst)
    lab = _tarjan(V, Fr.tolist(), Fc.tolist())
    return {"labels": torch.tensor(lab, dtype=torch.int32), "sccs": sum(lab[v] == v for v in range(1, V + 1))}


def _tarjan(V, Fr, Fc):
    index = [0] * (V + 1)
    low = [0] * (V + 1)
    lab = [0] * (V + 1)
    done = [False] * (V + 1)
    stack, n = [], 0
    for root in range(1, V + 1):
        if index[root]:
            continue
        n += 1
        index[root] = low[root] = n
        stack.append(root)
        work_list = [(root, Fr[root])]
        while work_list:
            v, i = work_list.pop()
            end, down = Fr[v + 1], False
            while i < end:
                w = Fc[i]
                i += 1
                if not index[w]:
                    n += 1
                    index[w] = low[w] = n
                    stack.append(w)
                    work_list.append((v, i))
                    work_list.append((w, Fr[w]))
                    down = True
                    break
                if not done[w] and index[w] < low[v]:
                    low[v] = index[w]
            if down:
                continue
            if low[v] == index[v]:
                members = []
                while True:
                    w = stack.pop()
                    done[w] = True
                    members.append(w)
                    if w == v:
                        break
                m = min(members)
                for w in members:
                    lab[w] = m
            if work_list:
                p = work_list[-1][0]
                if low[v] < low[p]:
                    low[p] = low[v]
    return lab
