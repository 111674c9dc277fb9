"""Workloads of the critical-path engine, timed through its public entry points.

Graphs are seeded layered timing DAGs of the kinds the benchmark and the
tests use: a share of the vertices are sources (level 0) and sinks (last
level), every other level holds an equal share, out-degrees are uniform
{1..4} or geometric, edges span one or a few levels, delays are uniform,
lognormal or 1.0, and vertex ids are a random permutation.

Kinds of case:
  query    one exact top-K path query on a resident graph, the K costs
           copied to host memory (reset, report_paths, get_slacks); options:
           level-order reorder, a share of the sinks as endpoints
  sfxt     the suffix forest alone, dist/succ/level copied to host memory
  noalloc  the suffix forest of a graph in the caller's device arrays
  batch    many designs, one query each, solved together
  serve    a saturated stream of endpoint-subset queries on resident graphs
  bvss     deviation edges leaving a set of source frontiers
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "gpu-cpg_amd"))
import cpgamd  # noqa: E402

SCALE = 10000


def device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the smallest design of a batch, queried alone: launches and latency
        {"name": "query_5k", "kind": "query", "n": 5003, "levels": 71, "deg": 4.0, "wgt": "lognormal", "k": 100},
        # the 50K-vertex, 120-level DAG of the tests at its K, long fan-in on the sinks
        {"name": "query_50k", "kind": "query", "n": 50000, "levels": 120, "deg": 0.0, "wgt": "uniform", "k": 10000},
        # unit delays (the text loader's ignore_wgts): ties everywhere
        {"name": "query_200k_unit", "kind": "query", "n": 200001, "levels": 447, "deg": 3.1, "wgt": "unit", "k": 20000},
        # the benchmark's headline: K = 1M on 1.5M vertices, level-order reorder
        {"name": "query_1500k_reorder", "kind": "query", "n": 1500000, "levels": 300, "deg": 2.7, "wgt": "lognormal",
         "k": 1000000, "reorder": True},
        # the same kind of graph as loaded (no reorder), an ordinary K
        {"name": "query_1100k", "kind": "query", "n": 1100003, "levels": 1049, "deg": 5.3, "wgt": "lognormal", "k": 30000},
        # a densified graph: a few long levels, mean out-degree 20
        {"name": "query_dense", "kind": "query", "n": 400000, "levels": 80, "deg": 20.0, "wgt": "lognormal", "k": 100000},
        # an endpoint subset on a deep graph with long fan-outs, as a served query asked alone
        {"name": "query_subset", "kind": "query", "n": 250007, "levels": 500, "deg": 27.0, "wgt": "lognormal", "k": 50000,
         "ends": 0.1},
        # the suffix forest alone
        {"name": "sfxt_700k", "kind": "sfxt", "n": 700001, "levels": 250, "deg": 3.3, "wgt": "lognormal"},
        # the suffix forest for a caller that may not allocate
        {"name": "noalloc_120k", "kind": "noalloc", "n": 120011, "levels": 346, "deg": 6.0, "wgt": "lognormal"},
        # designs of uneven size, one query each
        {"name": "batch_48", "kind": "batch", "designs": 48, "n_lo": 5000, "n_hi": 200000, "k_lo": 100, "k_hi": 100000},
        # resident graphs and a saturated stream of endpoint-subset queries
        {"name": "serve_24", "kind": "serve", "graphs": 3, "n_lo": 60000, "n_hi": 400000, "queries": 24, "k_lo": 1000,
         "k_hi": 300000},
        # deviation edges of consecutive-source frontiers
        {"name": "bvss_200k", "kind": "bvss", "n": 200000, "levels": 100, "deg": 20.0, "wgt": "lognormal", "fronts": 8,
         "span": 4096},
    ]


def log_between(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """Sizes log-uniform over the listed ranges; queries are most of the use."""
    kind = rng.choice(["query", "query", "query", "query", "sfxt", "noalloc", "batch", "serve", "bvss"])
    if kind == "batch":
        return {"kind": kind, "designs": rng.randint(3, 48), "n_lo": rng.randint(3000, 5000),
                "n_hi": rng.randint(20000, 200000), "k_lo": rng.randint(1, 100), "k_hi": rng.randint(1000, 100000)}
    if kind == "serve":
        return {"kind": kind, "graphs": rng.randint(1, 3), "n_lo": rng.randint(20000, 60000),
                "n_hi": rng.randint(80000, 400000), "queries": rng.randint(3, 24), "k_lo": rng.randint(100, 1000),
                "k_hi": rng.randint(5000, 300000)}
    deg = rng.choice([0.0, log_between(rng, 2.0, 6.0), log_between(rng, 6.0, 27.0)])
    n = int(log_between(rng, 4000, 1000000 if kind == "noalloc" else 1500000))
    if deg > 0:
        n = int(min(n, 8000000 / deg))
    # as deep as sqrt(n) levels, or as flat as the densified graph
    levels = max(12, int(math.sqrt(n) * rng.choice([1.0, rng.uniform(0.12, 1.0)])))
    case = {"kind": kind, "n": n, "levels": levels, "deg": round(deg, 2),
            "wgt": rng.choice(["lognormal", "lognormal", "uniform", "unit"])}
    if kind == "query":
        case["k"] = int(log_between(rng, 1, 1000000))
        if rng.random() < 0.25:
            case["reorder"] = True
        if rng.random() < 0.3:
            case["ends"] = round(log_between(rng, 0.01, 1.0), 3)
    if kind == "bvss":
        case["wgt"] = "lognormal"
        case["n"] = n = min(n, 300000)
        case["levels"] = min(levels, n // 20)
        case["fronts"] = rng.randint(1, 16)
        case["span"] = rng.randint(64, min(4096, n // 2))
    return case


# ----------------------------------------------------------------- graphs

def make_graph(n, levels, deg, wgt, gen, dev):
    """Edges of one DAG as device tensors in ascending source position: (u, v,
    w, ids, lstart).  u and v are positions in level order, ids[position] is
    the vertex id, lstart the levels' first positions.  deg 0: out-degree
    uniform {1..4}, spans {1..3} and an edge to a random sink; else geometric
    with that mean, nine spans in ten 1, the others {2..8}."""
    share = 0.01 if deg == 0 else 0.02
    ends = max(1, int(round(share * n)))
    mid = n - 2 * ends
    size = torch.full((levels,), mid // (levels - 2), dtype=torch.int64)
    size[1:1 + mid % (levels - 2)] += 1
    size[0] = size[-1] = ends
    lstart = torch.zeros(levels + 1, dtype=torch.int64)
    lstart[1:] = torch.cumsum(size, 0)
    size, first = size.to(dev), lstart.to(dev)
    level = torch.repeat_interleave(torch.arange(levels, device=dev), size)
    inner = n - ends  # every vertex but the sinks has fanouts

    def rand(k):
        return torch.rand(k, generator=gen, device=dev, dtype=torch.float64)

    def below(bound):  # an integer in [0, bound) for each entry of the tensor
        return torch.minimum((rand(bound.numel()) * bound).long(), bound - 1)

    if deg == 0:
        d = 1 + (rand(inner) * 4).long().clamp_(max=3)
    else:
        d = 1 + (torch.log1p(-rand(inner)) / math.log1p(-1.0 / deg)).long()
        d.clamp_(max=max(32, int(4 * deg)))
    u = torch.repeat_interleave(torch.arange(inner, device=dev), d)
    if deg == 0:
        span = 1 + (rand(u.numel()) * 3).long().clamp_(max=2)
    else:
        far = 2 + (rand(u.numel()) * 7).long().clamp_(max=6)
        span = torch.where(rand(u.numel()) < 0.9, torch.ones_like(far), far)
    tl = torch.clamp(level[u] + span, max=levels - 1)
    v = first[tl] + below(size[tl])
    if deg == 0:
        all_inner = torch.arange(inner, device=dev)
        u = torch.cat([u, all_inner])
        v = torch.cat([v, inner + below(torch.full_like(all_inner, ends))])
    bare = torch.ones(n, dtype=torch.bool, device=dev)
    bare[v] = False
    bare[:ends] = False
    b = bare.nonzero().flatten()  # no fanin yet: one from the level before
    u = torch.cat([u, first[level[b] - 1] + below(size[level[b] - 1])])
    v = torch.cat([v, b])
    key = torch.unique(u * n + v)  # no parallel edges
    u, v = key // n, key % n
    if wgt == "unit":
        w = torch.ones(u.numel(), device=dev)
    elif wgt == "uniform":
        w = (0.01 + 0.99 * rand(u.numel())).float()
    else:
        z = torch.randn(u.numel(), generator=gen, device=dev, dtype=torch.float64)
        w = torch.exp(-2.0 + 0.7 * z).float()
    ids = torch.randperm(n, generator=gen, device=dev)
    return u, v, w, ids, lstart.tolist()


def host_edges(graph):
    u, v, w, ids, _ = graph
    return (ids[u].int().cpu().numpy(), ids[v].int().cpu().numpy(), w.cpu().numpy())


def generator(seed, salt=0):
    gen = torch.Generator(device=device())
    gen.manual_seed((seed * 1000003 + salt) % (1 << 62))
    return gen


def case_graph(case, seed):
    return make_graph(case["n"], case["levels"], case["deg"], case["wgt"], generator(seed), device())


def endpoint_mask(n, graph, share, gen):
    """One byte per vertex id: the chosen sinks (at least one)."""
    _, _, _, ids, lstart = graph
    sinks = ids[lstart[-2]:]
    pick = torch.randperm(sinks.numel(), generator=gen, device=sinks.device)[:max(1, math.ceil(share * sinks.numel()))]
    mask = torch.zeros(n, dtype=torch.uint8, device=sinks.device)
    mask[sinks[pick]] = 1
    return mask


def members(case):
    """The sizes of a batch's designs, or of a served stream's graphs and
    queries."""
    rng = random.Random(case["n_lo"] * 1009 + case["k_hi"])

    def spread(lo, hi, count):  # log-even over the range, in random order
        out = [int(round(lo * (hi / lo) ** (i / max(1, count - 1)))) for i in range(count)]
        rng.shuffle(out)
        return out

    if case["kind"] == "batch":
        count = case["designs"]
        return [(n, int(math.sqrt(n)), 2.0 + 8.0 * rng.random(), k)
                for n, k in zip(spread(case["n_lo"], case["n_hi"], count), spread(case["k_lo"], case["k_hi"], count))]
    graphs = []
    for i in range(case["graphs"]):
        f = i / max(1, case["graphs"] - 1)
        n = int(case["n_lo"] * (case["n_hi"] / case["n_lo"]) ** f)
        graphs.append((n, int(math.sqrt(n)), (4.0, 27.0, 11.0)[i % 3]))
    queries = [(rng.randrange(case["graphs"]), k, max(0.01, 1.0 - rng.random()))
               for k in spread(case["k_lo"], case["k_hi"], case["queries"])]
    return graphs, queries


# -------------------------------------------------------- prepare and run

class Pinned(np.ndarray):
    """A pinned result buffer whose views keep the memory's owner alive."""

    def __array_finalize__(self, other):
        self.owner = getattr(other, "owner", None)


def pinned(k):
    owner = cpgamd.HostArray(k)
    out = owner.array.view(Pinned)
    out.owner = owner
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        b = cpgamd.Batch()
        ks = []
        for i, (n, levels, deg, k) in enumerate(members(case)):
            u, v, w = host_edges(make_graph(n, levels, deg, "lognormal", generator(seed, i), device()))
            b.add(n, u, v, w, k)
            ks.append(k)
        return {"kind": kind, "b": b, "ks": ks}
    if kind == "serve":
        graphs, queries = members(case)
        s = cpgamd.Server()
        made = []
        for i, (n, levels, deg) in enumerate(graphs):
            g = make_graph(n, levels, deg, "lognormal", generator(seed, i), device())
            s.add_graph(n, *host_edges(g))
            made.append(g)
        qs = [(gi, k, endpoint_mask(graphs[gi][0], made[gi], share, generator(seed, 100 + i)).cpu().numpy())
              for i, (gi, k, share) in enumerate(queries)]
        return {"kind": kind, "s": s, "qs": qs}
    graph = case_graph(case, seed)
    n = case["n"]
    if kind == "noalloc":
        u, v, w, ids, lstart = graph
        dev = u.device
        u, v = ids[u], ids[v]

        def csr(own):
            order = torch.argsort(own, stable=True)
            off = torch.zeros(n + 1, dtype=torch.int64, device=dev)
            off[1:] = torch.cumsum(torch.bincount(own, minlength=n), 0)
            return off.int(), order

        oadjp, _ = csr(u)
        iadjp, order = csr(v)
        iedge = torch.stack([u[order].int(), w[order].view(torch.int32)], 1).contiguous()
        sinks = torch.sort(ids[lstart[-2]:])[0].int()
        out = [torch.empty(n, dtype=torch.int32, device=dev) for _ in range(3)]
        return {"kind": kind, "n": n, "in": (oadjp, iadjp, iedge, sinks), "out": out}
    g = cpgamd.CpGen()
    g.load_edges(n, *host_edges(graph))
    if case.get("reorder"):
        g.set_csr_reorder(1)
    g.run_sfxt()  # the graph is resident from here on
    state = {"kind": kind, "g": g}
    if kind == "query":
        state["k"] = case["k"]
        state["out"] = pinned(case["k"])
        share = case.get("ends")
        state["mask"] = endpoint_mask(n, graph, share, generator(seed, 1)).cpu().numpy() if share else None
    elif kind == "bvss":
        g.bvss_build()
        rng = np.random.default_rng(seed)
        starts = rng.integers(0, n - case["span"], size=case["fronts"])
        state["src"] = np.concatenate([np.arange(s, s + case["span"], dtype=np.int32) for s in starts])
        state["ptr"] = np.arange(case["fronts"] + 1, dtype=np.int32) * np.int32(case["span"])
        room = int(1.5 * state["src"].size * mean_degree(case["deg"])) + 4096
        state["out"] = [np.zeros(room, np.int32) for _ in range(3)]
    return state


def address(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int))


def run(state):
    kind = state["kind"]
    if kind == "query":
        g, k = state["g"], state["k"]
        g.reset()
        g.report_paths(k, endpoint_mask=state["mask"])
        return g.get_slacks(k, out=state["out"])
    if kind == "sfxt":
        g = state["g"]
        g.reset()
        g.run_sfxt()
        return g.sfxt()
    if kind == "noalloc":
        oadjp, iadjp, iedge, sinks = state["in"]
        dist, succ, level = state["out"]
        levels = cpgamd.lib().cpg_sfxt_noalloc(
            state["n"], oadjp.data_ptr(), iadjp.data_ptr(), iedge.data_ptr(), sinks.data_ptr(), sinks.numel(),
            dist.data_ptr(), succ.data_ptr(), level.data_ptr(), torch.cuda.current_stream().cuda_stream)
        if levels < 0:
            raise RuntimeError(cpgamd.lib().cpg_last_error().decode())
        return levels, dist, succ, level
    if kind == "batch":
        state["b"].run()
        return [state["b"].get_slacks(q, k) for q, k in enumerate(state["ks"])]
    if kind == "serve":
        s = state["s"]
        ids = [s.submit(gi, k, mask) for gi, k, mask in state["qs"]]
        while s.step() > 0:
            pass
        s.poll()
        costs = [s.get_slacks(q, k) for q, (_, k, _) in zip(ids, state["qs"])]
        for q in ids:
            s.release(q)
        return costs
    g, ptr, src, (of, ou, ov) = state["g"], state["ptr"], state["src"], state["out"]
    found = g.L.cpg_bvss_discover(g.h, len(ptr) - 1, address(ptr), address(src), 0, 4, address(of), address(ou),
                                  address(ov), len(of))
    if found < 0:
        raise RuntimeError(g.L.cpg_last_error().decode())
    return found, of, ou, ov


# ------------------------------------------------------------------- work

def mean_degree(deg):
    return 3.5 if deg == 0 else deg


def work(case):
    """The graph read once (fanout offsets, heads and weights) and the result
    written once; each edge is relaxed once (an add and a minimum)."""
    kind = case["kind"]
    if kind == "batch":
        mem = members(case)
        nodes = sum(n for n, _, _, _ in mem)
        edges = sum(n * d for n, _, d, _ in mem)
        return {"bytes": 4 * nodes + 8 * edges + 4 * sum(k for _, _, _, k in mem), "flops": 2 * edges}
    if kind == "serve":
        graphs, queries = members(case)
        total = edges = 0
        for gi, k, _ in queries:
            n, _, d = graphs[gi]
            total += 4 * n + 8 * n * d + n + 4 * k
            edges += n * d
        return {"bytes": total, "flops": 2 * edges}
    n, m = case["n"], case["n"] * mean_degree(case["deg"])
    if kind == "bvss":
        found = case["fronts"] * case["span"] * mean_degree(case["deg"])
        return {"bytes": 4 * case["fronts"] * case["span"] + 20 * found, "flops": found}
    out = 4 * case["k"] if kind == "query" else 12 * n
    return {"bytes": 4 * n + 8 * m + out + (n if case.get("ends") else 0), "flops": 2 * m}


# ------------------------------------------------------------------ exact

def forest(graph, n, mask=None):
    """Suffix forest in 64 bits, by level-order position: int-scaled distances
    (weights scaled and cut to integers in single precision, as the format
    defines them), successors (largest id at the minimum), -1 / a large
    distance where no chosen sink is reached."""
    u, v, w, ids, lstart = graph
    dev = u.device
    far = torch.iinfo(torch.int64).max // 4
    dist = torch.full((n,), far, dtype=torch.int64, device=dev)
    succ = torch.full((n,), -1, dtype=torch.int64, device=dev)
    sinks = torch.arange(lstart[-2], n, device=dev)
    if mask is not None:
        sinks = sinks[mask[ids[sinks]] != 0]
    dist[sinks] = 0
    wi = (w * float(SCALE)).long()
    pos_of = torch.empty_like(ids)
    pos_of[ids] = torch.arange(n, device=dev)
    cut = torch.searchsorted(u, torch.tensor(lstart, device=dev)).tolist()
    for lv in range(len(lstart) - 3, -1, -1):
        a, b = cut[lv], cut[lv + 1]
        if a == b:
            continue
        eu, ev = u[a:b], v[a:b]
        cand = torch.clamp(dist[ev] + wi[a:b], max=far)
        dist.scatter_reduce_(0, eu, cand, "amin")
        best = (cand == dist[eu]) & (cand < far)
        top = torch.full((lstart[lv + 1] - lstart[lv],), -1, dtype=torch.int64, device=dev)
        top.scatter_reduce_(0, eu[best] - lstart[lv], ids[ev[best]], "amax")
        succ[lstart[lv]:lstart[lv + 1]] = torch.where(top >= 0, pos_of[top.clamp(min=0)], top)
    return dist, succ, far


def exact_costs(graph, n, k, mask=None):
    """The k smallest path costs of a query in 64 bits: roots (sources, with
    the initial split's truncation of ties), and every path that takes
    deviation edges off a suffix chain; all paths up to a cost are listed, and
    the cost is widened until there are k."""
    u, v, w, ids, lstart = graph
    dev = u.device
    dist, succ, far = forest(graph, n, mask)
    df = dist.double() / SCALE
    use = (dist[v] < far) & (dist[u] < far) & (succ[u] != v)
    du, dv = u[use], v[use]
    delta = df[dv] + w[use].double() - df[du]
    order = torch.argsort(delta, stable=True)
    order = order[torch.argsort(du[order], stable=True)]
    du, dv, delta = du[order], dv[order], delta[order]
    first = torch.zeros(n + 1, dtype=torch.int64, device=dev)
    first[1:] = torch.cumsum(torch.bincount(du, minlength=n), 0)
    has = first[1:] > first[:-1]
    best = torch.full((n,), math.inf, dtype=torch.float64, device=dev)
    best[has] = delta[first[:-1][has]]
    low = best.clone()  # the smallest deviation anywhere on the chain from here
    for lv in range(len(lstart) - 3, -1, -1):
        a, b = lstart[lv], lstart[lv + 1]
        s = succ[a:b]
        low[a:b] = torch.where(s >= 0, torch.minimum(low[a:b], low[s.clamp(min=0)]), low[a:b])
    src = torch.arange(lstart[1], device=dev)
    src = src[torch.argsort(ids[src])]
    src = src[dist[src] < far]
    if src.numel() == 0 or k == 0:
        return np.zeros(0)
    split_at = 0.005 * src.numel()
    rank = min(int(np.float32(0.005) * np.float32(src.numel())), src.numel() - 1)
    split = torch.sort(dist[src])[0][rank]
    under = dist[src] <= split
    src = src[~under | (torch.cumsum(under.long(), 0) <= int(np.float32(split_at) + 1))]
    roots = df[src]

    def paths(bound, most):
        keep = roots <= bound
        c, x, j = roots[keep], src[keep], first[:-1][src[keep]]
        got = [c]
        total = c.numel()
        while c.numel():
            at = j.clamp(max=max(0, delta.numel() - 1))
            cc = c + delta[at] if delta.numel() else torch.full_like(c, math.inf)
            take = (j < first[x + 1]) & (cc <= bound)
            hc, hx = cc[take], dv[at[take]]
            got.append(hc)
            total += hc.numel()
            if total > most:
                return None
            nx = succ[x]
            on = ~take & (nx >= 0)
            on &= c + low[nx.clamp(min=0)] <= bound
            new = c + 0
            down = c[on]
            live = hc + low[hx] <= bound
            c = torch.cat([new[take], down, hc[live]])
            j = torch.cat([j[take] + 1, first[nx[on]], first[hx[live]]])
            x = torch.cat([x[take], nx[on], hx[live]])
        return torch.cat(got)

    base = float(roots.min())
    lo, hi, gap = 0.0, None, max(float(roots.median()) - base, 1e-3 * max(base, 1e-3))
    last = None
    for _ in range(60):
        found = paths(base + gap, max(4 * k, 1 << 16) + roots.numel())
        if found is None:
            hi = gap
        elif found.numel() >= k:
            return torch.sort(found)[0][:k].cpu().numpy()
        else:
            if last is not None and hi is None and found.numel() == last and gap > 1e6:
                return torch.sort(found)[0].cpu().numpy()  # fewer than k paths in all
            last = found.numel()
            lo = gap
        gap = gap * 1.6 if hi is None else 0.5 * (lo + hi)
    return None


def exact(case, seed):
    """Costs in 64 bits; whole-number results have none.  Unit delays put far
    more than k paths at one cost, so they are not listed."""
    kind = case["kind"]
    if kind == "query" and case["wgt"] != "unit":
        graph = case_graph(case, seed)
        share = case.get("ends")
        mask = endpoint_mask(case["n"], graph, share, generator(seed, 1)) if share else None
        return exact_costs(graph, case["n"], case["k"], mask)
    if kind == "batch":
        return [exact_costs(make_graph(n, levels, deg, "lognormal", generator(seed, i), device()), n, k)
                for i, (n, levels, deg, k) in enumerate(members(case))]
    if kind == "serve":
        graphs, queries = members(case)
        made = [make_graph(n, levels, deg, "lognormal", generator(seed, i), device())
                for i, (n, levels, deg) in enumerate(graphs)]
        return [exact_costs(made[gi], graphs[gi][0], k,
                            endpoint_mask(graphs[gi][0], made[gi], share, generator(seed, 100 + i)))
                for i, (gi, k, share) in enumerate(queries)]
    return None
