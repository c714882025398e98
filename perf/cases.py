"""Performance cases: calls of the public Python API over the sizes and graphs
that its users run, from one small graph whose call is all latency to the
largest configured ones.

Graphs are generated on the GPU with torch from the seed alone (Erdos-Renyi,
R-MAT with quadrant probabilities 0.57 / 0.19 / 0.19 / 0.05 and Chung-Lu with
exponent 2.1, the three families of the benchmark and the tests, and blocks
joined by R-MAT edges where clusters are looked for), symmetrised,
deduplicated and without self-loops, with a fixed number of edges, and handed
to the framework as host CSR arrays.  `listed()` says what each case stands for; `draw()` gives further
sizes of the same calls.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from acctricnt_amd import cn, serve
from acctricnt_amd.graph import CSRGraph

# Exact counts are taken by listing, for every edge, its shorter list: at most
# this many list entries in all (a few seconds on the GPU).
EXACT_WEDGES = 2_000_000_000
_PASS = 1 << 26  # entries handled at a time

_context = None


def _ctx():
    """The process's one context, as a program holds it."""
    global _context
    if _context is None:
        _context = cn.Context(0)
    return _context


def listed():
    return [
        # a whole call on one small graph (the ER fixture's size): launches,
        # copies and waits, hardly any counting
        {"name": "small-count-read", "call": "count_read", "graph": "er", "n": 16384, "deg": 16.0},
        # the smallest call: the triangle total of a graph of a few thousand vertices
        {"name": "small-triangles", "call": "triangles", "graph": "chung_lu", "n": 3001, "deg": 24.0},
        # an ordinary graph of odd size, counts left in HBM in the raw format
        # (for a consumer on the GPU)
        {"name": "medium-count", "call": "count", "graph": "rmat", "n": 100003, "deg": 24.0, "raw": True},
        # the headline workload: R-MAT scale 22 (edge factor 16 before duplicates go), counts left in HBM
        {"name": "large-count", "call": "count", "graph": "rmat", "n": 1 << 22, "deg": 30.5, "raw": False},
        # the other large family: a power law with hubs of hundreds of thousands of neighbors
        {"name": "hub-count", "call": "count", "graph": "chung_lu", "n": 3000017, "deg": 32.0, "raw": False},
        # triangle counting alone (main_triangle_count) on a large resident graph
        {"name": "large-triangles", "call": "triangles", "graph": "rmat", "n": 1 << 21, "deg": 32.0},
        # many graphs in one packed CSR, the pass captured once and replayed,
        # per-graph totals read back
        {"name": "batch-replay", "call": "replay", "graph": "batch", "graphs": 512, "n_lo": 256, "n_hi": 65536},
        # one-shot use: host arrays in, counts in host memory out
        {"name": "upload-count-read", "call": "upload_count", "graph": "rmat", "n": 500009, "deg": 32.0},
        # the SCAN program (main_scanxp): a graph as generated, relabelled at
        # upload, counted and clustered, labels read
        {"name": "upload-scan", "call": "upload_scan", "graph": "communities", "n": 262144, "deg": 28.0, "eps": "0.4", "mu": 5},
        # further SCAN queries on a resident graph whose counts are there
        {"name": "scan-query", "call": "scan", "graph": "rmat", "n": 1 << 20, "deg": 32.0, "eps": "0.2", "mu": 5},
        # a burst of queries to the serving loop over a few resident graphs
        {"name": "serve-burst", "call": "serve", "graph": "communities", "n": 131072, "deg": 28.0, "graphs": 5, "queries": 24},
        # the reference's bitmap method, selected by name
        {"name": "bitmap-count", "call": "bitmap", "graph": "rmat", "n": 262144, "deg": 32.0, "raw": False},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["count_read", "triangles", "count", "count", "count", "triangles", "replay", "upload_count",
                       "upload_scan", "scan", "serve", "bitmap"])
    case = {"call": call, "graph": rng.choice(["er", "rmat", "chung_lu"]), "deg": round(rng.uniform(8.0, 32.0), 1)}
    if call == "replay":
        return {"call": call, "graph": "batch", "graphs": rng.randint(60, 512), "n_lo": 256,
                "n_hi": _log_uniform(rng, 4096, 65536)}
    if call in ("scan", "upload_scan", "serve"):
        case["graph"] = rng.choice(["rmat", "communities"])
    lo, hi = {"count_read": (4000, 60000), "triangles": (3000, 2000000), "count": (30000, 3000000),
              "upload_count": (30000, 500000), "upload_scan": (30000, 262144), "scan": (30000, 1 << 20),
              "serve": (20000, 131072), "bitmap": (30000, 262144)}[call]
    case["n"] = _log_uniform(rng, lo, hi)
    if call in ("count", "bitmap"):
        case["raw"] = rng.random() < 0.5
    if call in ("scan", "upload_scan"):
        case.update(eps="0.%d" % rng.randint(1, 5), mu=rng.choice([2, 5, 10]))
    if call == "serve":
        case.update(graphs=rng.randint(2, 6), queries=rng.randint(8, 28))
    return case


# ---------------------------------------------------------------- graphs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _sample_er(gen, n, samples):
    return (torch.randint(0, n, (samples,), generator=gen, device="cuda"),
            torch.randint(0, n, (samples,), generator=gen, device="cuda"))


def _sample_rmat(gen, scale, samples):
    """Endpoints over 2^scale ids; scale may be one number or one per sample."""
    u = torch.zeros(samples, dtype=torch.int64, device="cuda")
    v = torch.zeros_like(u)
    top = int(scale.max()) if torch.is_tensor(scale) else scale
    for level in range(top):
        r = torch.rand(samples, generator=gen, device="cuda")
        ub = r >= 0.76
        vb = ((r >= 0.57) & ~ub) | (r >= 0.95)
        if torch.is_tensor(scale):
            on = level < scale
            u = torch.where(on, 2 * u + ub, u)
            v = torch.where(on, 2 * v + vb, v)
        else:
            u = 2 * u + ub
            v = 2 * v + vb
    return u, v


def _sample_chung_lu(gen, n, samples):
    w = (torch.arange(n, dtype=torch.float64, device="cuda") + 1.0).pow(-1.0 / 1.1)
    w = w.clamp_(max=float(w.sum()) * n / (16.0 * samples))  # expected degrees up to about n / 8
    c = torch.cumsum(w, 0)
    ends = []
    for _ in range(2):
        r = torch.rand(samples, dtype=torch.float64, generator=gen, device="cuda") * c[-1]
        ends.append(torch.searchsorted(c, r).clamp_(max=n - 1))
    return ends


def _sample_communities(gen, n, samples):
    """Seven of ten edges inside blocks of consecutive ids (sizes 12 to 83 by
    turns), the rest R-MAT edges: clusters joined by hubs."""
    size = 12 + (torch.arange(n // 12 + 1, device="cuda") * 29) % 72
    ends = torch.cumsum(size, 0)
    inside = samples * 7 // 10
    u = torch.randint(0, n, (inside,), generator=gen, device="cuda")
    block = torch.searchsorted(ends, u, right=True)
    v = ends[block] - size[block] + (torch.rand(inside, generator=gen, device="cuda") * size[block]).long()
    ru, rv = _sample_rmat(gen, max(1, math.ceil(math.log2(n))), samples - inside)
    return torch.cat([u, ru]), torch.cat([v, rv])


_SAMPLE = {"er": _sample_er, "chung_lu": _sample_chung_lu, "communities": _sample_communities,
           "rmat": lambda gen, n, samples: _sample_rmat(gen, max(1, math.ceil(math.log2(n))), samples)}


def _edge_keys(n, u, v):
    """Distinct undirected edges without self-loops, as keys n * smaller + larger."""
    keep = (u != v) & (u < n) & (v < n)
    u, v = u[keep], v[keep]
    return torch.unique(torch.minimum(u, v) * n + torch.maximum(u, v))


def _slots(gen, n, keys, edges):
    """The sorted slots (source, target) of `edges` edges, picked at random from the distinct ones."""
    keys = keys[torch.randperm(keys.numel(), generator=gen, device="cuda")[:edges]]
    u, v = keys // n, keys % n
    key = torch.sort(torch.cat([u * n + v, v * n + u])).values
    return key // n, key % n


def _by_degree(n, src, dst):
    """Ids by degree, descending, ties by id: the relabel the graphs are loaded with."""
    order = torch.argsort(torch.bincount(src, minlength=n), descending=True, stable=True)
    new = torch.empty_like(order)
    new[order] = torch.arange(n, device="cuda")
    key = torch.sort(new[src] * n + new[dst]).values
    return key // n, key % n


def _csr(n, src, dst):
    off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.cumsum(torch.bincount(src, minlength=n), 0)
    return CSRGraph(off.cpu().numpy().astype(np.uint32), dst.to(torch.int32).cpu().numpy())


def _graph_slots(case, seed):
    """n, then the source and target of every slot: exactly n * deg / 2 edges."""
    gen = _generator(seed)
    n, edges = case["n"], int(case["n"] * case["deg"] / 2)
    keys = torch.empty(0, dtype=torch.int64, device="cuda")
    while keys.numel() < edges:
        u, v = _SAMPLE[case["graph"]](gen, n, max(1024, int(1.1 * edges)))
        keys = torch.unique(torch.cat([keys, _edge_keys(n, u, v)])) if keys.numel() else _edge_keys(n, u, v)
    src, dst = _slots(gen, n, keys, edges)
    if case["call"] != "upload_scan":  # that call relabels on the device
        src, dst = _by_degree(n, src, dst)
    return n, src, dst


def _batch_sizes(case):
    """Vertex counts (log-uniform), average degrees before duplicates go
    (uniform in [4, 64]) and families of the packed graphs."""
    rng = np.random.default_rng(2024)
    k = case["graphs"]
    ns = np.exp(rng.uniform(math.log(case["n_lo"]), math.log(case["n_hi"]), k)).round().astype(np.int64)
    return ns, rng.uniform(4.0, 64.0, k), rng.integers(0, 3, k)


def _batch_slots(case, seed):
    """The packed mix, a third of the graphs of each family; 0.6 of the
    sampled edges in all, a number that the distinct ones always reach."""
    ns, deg, family = _batch_sizes(case)
    vertex_off = np.zeros(case["graphs"] + 1, np.int64)
    np.cumsum(ns, out=vertex_off[1:])
    n = int(vertex_off[-1])
    samples = (ns * deg / 2).astype(np.int64)
    gen = _generator(seed)
    keys = []
    for f in range(3):
        which = np.nonzero(family == f)[0]
        if not which.size:
            continue
        reps = torch.from_numpy(samples[which]).cuda()
        n_of = torch.repeat_interleave(torch.from_numpy(ns[which]).cuda(), reps)
        base = torch.repeat_interleave(torch.from_numpy(vertex_off[which]).cuda(), reps)
        total = int(samples[which].sum())
        if f == 0:
            u, v = ((torch.rand(total, dtype=torch.float64, generator=gen, device="cuda") * n_of).long() for _ in range(2))
        elif f == 1:
            u, v = _sample_rmat(gen, torch.ceil(torch.log2(n_of.double())).long(), total)
        else:
            # ids by inverting the power law's continuous distribution function
            top = n_of.double().pow(1.0 / 11.0)
            u, v = ((1.0 + torch.rand(total, dtype=torch.float64, generator=gen, device="cuda") * (top - 1.0)).pow(11.0)
                    .long().sub_(1).clamp_(min=0) for _ in range(2))
        keep = (u < n_of) & (v < n_of)
        keys.append(_edge_keys(n, (u + base)[keep], (v + base)[keep]))
    src, dst = _slots(gen, n, torch.sort(torch.cat(keys)).values, _batch_edges(case))
    return n, src, dst, vertex_off.astype(np.uint32)


def _batch_edges(case):
    ns, deg, _ = _batch_sizes(case)
    return int(0.6 * (ns * deg / 2).sum())


# ---------------------------------------------------------------- the calls
class _DeviceArray:
    """A resident graph's counts for torch.as_tensor, which holds this object
    (and with it the graph, whose memory the tensor reads) for the tensor's life."""

    def __init__(self, rg):
        self.graph = rg
        self.__cuda_array_interface__ = {"shape": (rg.m,), "typestr": "<i4", "data": (rg.device_counts_ptr(), False),
                                         "version": 2}


def _counts_view(rg):
    return torch.as_tensor(_DeviceArray(rg), device="cuda")


def _serve_plan(case):
    """(graph, eps, mu) of every query, over the serving benchmark's grid."""
    rng = np.random.default_rng(2024)
    return [(int(rng.integers(case["graphs"])), "0.%d" % rng.integers(1, 10), int(rng.choice([2, 5, 10, 20])))
            for _ in range(case["queries"])]


def prepare(case, seed):
    ctx = _ctx()
    call = case["call"]
    state = {"case": case, "ctx": ctx}
    if call == "replay":
        n, src, dst, vertex_off = _batch_slots(case, seed)
        rg = ctx.upload(_csr(n, src, dst))
        rg.set_partition(vertex_off)
        rg.capture()
        state.update(rg=rg, counts=_counts_view(rg))
    elif call == "serve":
        sv = serve.Server(ctx, slots=32)
        sizes = [max(1000, case["n"] >> (i % 3)) + i for i in range(case["graphs"])]
        gids = [sv.add_graph(_csr(*_graph_slots({**case, "n": m}, seed * 8 + i))) for i, m in enumerate(sizes)]
        state.update(server=sv, plan=[(gids[k], eps, mu) for k, eps, mu in _serve_plan(case)])
    else:
        g = _csr(*_graph_slots(case, seed))
        if call in ("upload_count", "upload_scan"):
            state["graph"] = g
        else:
            rg = state["rg"] = ctx.upload(g)
            if call in ("count", "bitmap"):
                state["counts"] = _counts_view(rg)
            elif call == "scan":
                rg.compute()
                state["ws"] = rg.scan_workspace()
    return state


def run(state):
    case = state["case"]
    call = case["call"]
    if call == "count":
        state["rg"].compute(raw=case["raw"])
        return state["counts"]
    if call == "bitmap":
        state["rg"].compute("bitmap", raw=case["raw"])
        return state["counts"]
    if call == "count_read":
        return state["rg"].count_all_edges()
    if call == "triangles":
        return state["rg"].triangle_total()
    if call == "replay":
        state["rg"].replay()
        return state["counts"], state["rg"].graph_totals()
    if call == "upload_count":
        with state["ctx"].upload(state["graph"]) as rg:
            return rg.count_all_edges()
    if call == "upload_scan":
        with state["ctx"].upload(state["graph"], relabel=True) as rg, rg.scan_workspace() as ws:
            ws.run(case["eps"], case["mu"])
            return ws.results(core_count=True)
    if call == "scan":
        state["ws"].run(case["eps"], case["mu"])
        return state["ws"].results(core_count=True)
    sv = state["server"]
    tickets = [sv.submit(gid, eps, mu) for gid, eps, mu in state["plan"]]
    out = []
    for t in tickets:
        sv.wait(t)
        r = sv.result(t)
        out.append((r["label"], r["cluster_id"]))
        sv.release(t)
    return out


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Bytes of one pass (slots = directed edges): the graph read once and the
    results written once."""
    call = case["call"]
    if call == "replay":
        n, slots = int(_batch_sizes(case)[0].sum()), 2.0 * _batch_edges(case)
    else:
        n, slots = case["n"], case["n"] * case["deg"]
    graph = 4.0 * (n + 1) + 4.0 * slots
    if call == "triangles":
        return {"bytes": graph + 8, "flops": 0}
    if call in ("scan", "upload_scan"):  # labels, cluster ids and core counts; the query also reads the counts
        return {"bytes": graph + 12.0 * n + (4.0 * slots if call == "scan" else 0), "flops": 0}
    if call == "serve":  # a label byte and a cluster id per vertex and query
        return {"bytes": 5.0 * case["queries"] * n / 2, "flops": 0}
    return {"bytes": graph + 4.0 * slots, "flops": 0}


# ---------------------------------------------------------------- the counts by definition
def _exact_counts(n, src, dst):
    """|N(u) ∩ N(v)| of every slot: the entries of the shorter list of each
    edge looked up among all slots.  None when that is too many entries."""
    key = src * n + dst
    deg = torch.bincount(src, minlength=n)
    off = torch.cumsum(deg, 0) - deg
    up = torch.nonzero(src < dst).flatten()
    u, v = src[up], dst[up]
    swap = deg[u] > deg[v]
    short, other = torch.where(swap, v, u), torch.where(swap, u, v)
    ends = torch.cumsum(deg[short], 0)
    if ends.numel() == 0 or int(ends[-1]) > EXACT_WEDGES:
        return None if ends.numel() else torch.zeros_like(src)
    got = torch.zeros_like(u)
    lo = 0
    while lo < u.numel():
        start = int(ends[lo - 1]) if lo else 0
        hi = max(lo + 1, int(torch.searchsorted(ends, start + _PASS, right=True)))
        length = deg[short[lo:hi]]
        edge = torch.repeat_interleave(torch.arange(lo, hi, device="cuda"), length)
        first = torch.repeat_interleave(torch.cumsum(length, 0) - length, length)
        w = dst[off[short[edge]] + torch.arange(edge.numel(), device="cuda") - first]
        wanted = other[edge] * n + w
        hit = key[torch.searchsorted(key, wanted).clamp_(max=key.numel() - 1)] == wanted
        got += torch.bincount(edge[hit], minlength=u.numel())
        lo = hi
    counts = torch.empty_like(src)
    counts[up] = got
    counts[torch.searchsorted(key, v * n + u)] = got
    return counts


def exact(case, seed):
    """Counts and totals in 64-bit integers for the counting calls (SCAN's
    results are labels, not computed numbers)."""
    call = case["call"]
    if call in ("scan", "upload_scan", "serve"):
        return None
    if call == "replay":
        n, src, dst, vertex_off = _batch_slots(case, seed)
    else:
        n, src, dst = _graph_slots(case, seed)
    counts = _exact_counts(n, src, dst)
    if counts is None:
        return None
    total = int(counts.sum()) // 6
    if call == "triangles":
        return total
    if call == "replay":
        graph_of = torch.searchsorted(torch.from_numpy(vertex_off[1:].astype(np.int64)).cuda(), src, right=True)
        totals = torch.zeros(case["graphs"], dtype=torch.int64, device="cuda").index_add_(0, graph_of, counts) // 6
        return counts + 2, totals
    counts = counts if case.get("raw") else counts + 2
    return (counts, total) if call in ("count_read", "upload_count") else counts
