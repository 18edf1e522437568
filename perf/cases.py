"""The workloads this library's speed is judged on, through its Python entry points.

A case names one workload: a seeded random graph (or several) and the queries a program runs on
it.  `prepare` builds what such a program holds before the call (resident graphs, a prepared batch,
a running server, or a host edge list), `run` makes one pass and returns its counts.

Graphs are generated here with torch: R-MAT (a/b/c/d = 0.57/0.19/0.19/0.05, any vertex count),
Erdos-Renyi, Barabasi-Albert and Chung-Lu, the families of the benchmark's workloads.
"""
import gc
import math

import numpy as np
import torch

import jupiter_amd as J

DEV = "cuda" if torch.cuda.is_available() else "cpu"

# P4, P6, P8 and P10 pair up or intersect again every member of an edge's common neighbourhood, so
# they are asked of small graphs; the clique, diamond and triangle-based ids of large ones.
TABLE4 = ("P2", "P5", "P9", "P13", "P14")  # the reference's run_table4.sh
MOTIFS = ("I_C4", "I_DIAMOND", "I_TAILTRI", "I_STAR3")
SMALL_SET = ("TC", "P13", "P1", "P2")  # the batched workload's patterns
# largest log2 of the vertex count a drawn query of the pattern gets, and the smallest
RANGE = {"TC": (8, 22), "P13": (8, 22), "P14": (8, 22), "P15": (8, 16.5), "P16": (8, 12),
         "P1": (8, 18.5), "P2": (8, 20), "P3": (8, 19), "P5": (8, 17.7), "P7": (8, 17.5), "P9": (8, 18),
         "P11": (8, 18), "P12": (8, 17.5), "P4": (8, 14.3), "P6": (8, 10.8), "P8": (8, 12), "P10": (8, 10.3)}
SERVED = ("TC", "P1", "P2", "P3", "P5", "P7", "P9", "P11", "P12", "P13", "P14")


def listed():
    return [
        # the smallest calls: the batched workload's patterns as plain calls on its smallest graph,
        # where launches and host work count
        {"name": "plain_er1000", "kind": "query", "graph": "er", "n": 1000, "ef": 8, "patterns": ",".join(SMALL_SET),
         "part": 0, "parts": 1},
        # triangle count of a mid-sized graph, one range: launch-bound latency
        {"name": "tc_rmat14", "kind": "query", "graph": "rmat", "n": 1 << 14, "ef": 16, "patterns": "TC", "part": 0,
         "parts": 1},
        # the benchmark's step: 4- and 5-cliques over the heaviest quarter of the roots of R-MAT 22
        {"name": "cliques_rmat22_q0", "kind": "query", "graph": "rmat", "n": 1 << 22, "ef": 16,
         "patterns": "P13,P14", "part": 0, "parts": 4},
        # 6-cliques of a mid-sized graph (the deeper clique ids)
        {"name": "p15_rmat16", "kind": "query", "graph": "rmat", "n": 1 << 16, "ef": 16, "patterns": "P15", "part": 0,
         "parts": 1},
        # 4-cycles of the smallest graph size of the serving workload
        {"name": "p1_rmat18", "kind": "query", "graph": "rmat", "n": 1 << 18, "ef": 16, "patterns": "P1", "part": 0,
         "parts": 1},
        # a triangle-based 5-vertex pattern of the reference's result table, same size
        {"name": "p5_rmat18", "kind": "query", "graph": "rmat", "n": 1 << 18, "ef": 16, "patterns": "P5", "part": 0,
         "parts": 1},
        # two of the patterns with a second intersection inside the nest, at the size of the test graphs
        {"name": "p4_rmat14", "kind": "query", "graph": "rmat", "n": 1 << 14, "ef": 16, "patterns": "P4", "part": 0,
         "parts": 1},
        {"name": "p8_rmat12", "kind": "query", "graph": "rmat", "n": 1 << 12, "ef": 16, "patterns": "P8", "part": 0,
         "parts": 1},
        # vertex-induced 4-vertex motifs of the 3.8M-vertex power-law graph
        {"name": "motifs_chunglu", "kind": "query", "graph": "chunglu", "n": 3800000, "ef": 4.34,
         "patterns": ",".join(MOTIFS), "part": 0, "parts": 1},
        # many small graphs, one pattern each, in a prepared batch that is replayed
        {"name": "batch_96", "kind": "batch", "graphs": 96, "n_min": 1000, "n_max": 131072, "replay": True},
        # one dataset of the reference's result table from its edge list: build the resident graph,
        # count, let it go
        {"name": "table4_edges_rmat16", "kind": "edges", "graph": "rmat", "n": 1 << 16, "ef": 16,
         "patterns": ",".join(TABLE4)},
        # concurrent requests on resident graphs through the server
        {"name": "serve_48", "kind": "serve", "graphs": 8, "n_min": 1 << 12, "n_max": 1 << 16, "requests": 48},
    ]


def _log_size(rng, lo, hi):
    return int(2.0 ** rng.uniform(lo, hi))


def draw(rng):
    kind = rng.choice(["small", "clique", "clique", "sym", "sym", "nest", "nest", "motifs", "batch", "edges", "serve"])
    if kind == "small":
        p = rng.sample(sorted(SMALL_SET), rng.randint(1, 4))
        return {"kind": "query", "graph": rng.choice(["er", "ba", "rmat"]), "n": _log_size(rng, 8, 13),
                "ef": rng.randint(4, 32), "patterns": ",".join(p), "part": 0, "parts": 1}
    if kind in ("clique", "sym", "nest"):
        p = rng.choice({"clique": ["TC", "P13", "P14", "P15", "P16"], "nest": ["P4", "P6", "P8", "P10"],
                        "sym": ["P1", "P2", "P3", "P5", "P7", "P9", "P11", "P12"]}[kind])
        lo, hi = RANGE[p]
        n = _log_size(rng, lo if kind == "nest" else lo + 2, hi)
        parts = 4 if n > (1 << 20) else rng.choice([1, 1, 1, 4])
        return {"kind": "query", "graph": "rmat", "n": n, "ef": rng.randint(6, 16), "patterns": p,
                "part": rng.randrange(parts), "parts": parts}
    if kind == "motifs":
        return {"kind": "query", "graph": "chunglu", "n": _log_size(rng, 14, 21.8), "ef": round(rng.uniform(3, 5), 2),
                "patterns": ",".join(MOTIFS), "part": 0, "parts": 1}
    if kind == "batch":
        return {"kind": "batch", "graphs": rng.randint(16, 96), "n_min": 1000, "n_max": _log_size(rng, 12, 17),
                "replay": rng.random() < 0.6}
    if kind == "edges":
        return {"kind": "edges", "graph": "rmat", "n": _log_size(rng, 10, 16.5), "ef": rng.randint(6, 16),
                "patterns": ",".join(sorted(rng.sample(TABLE4, rng.randint(2, 5))))}
    return {"kind": "serve", "graphs": rng.randint(4, 12), "n_min": 1 << 10, "n_max": _log_size(rng, 13, 16),
            "requests": rng.randint(16, 56)}


# ---------------------------------------------------------------------------
# Graphs: undirected edge lists (int32 host arrays, duplicates and loops among them, as read from a file)


def _rand(g, size):
    return torch.rand(size, generator=g, device=DEV, dtype=torch.float32)


def _rmat_edges(n, m, g):
    bits = max(1, (n - 1).bit_length())
    u = torch.zeros(m, dtype=torch.int64, device=DEV)
    v = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(bits):
        x = _rand(g, m)
        u = (u << 1) | (x >= 0.76)
        v = (v << 1) | (((x >= 0.57) & (x < 0.76)) | (x >= 0.95))
    if n != 1 << bits:  # spread the 2^bits ids over n
        u, v = (u * n) >> bits, (v * n) >> bits
    return u, v


def _er_edges(n, m, g):
    return tuple(torch.randint(0, n, (m,), generator=g, device=DEV) for _ in range(2))


def _ba_edges(n, m, g):
    """m attachments per vertex: an edge's target is the endpoint in a uniformly chosen earlier slot."""
    e = n * m
    src = torch.arange(e, device=DEV) // m
    pick = (torch.rand(e, generator=g, device=DEV, dtype=torch.float64) * (2 * torch.arange(e, device=DEV) + 1)).long()
    slot = pick
    while bool((slot & 1).any()):  # odd slots are targets themselves: follow them
        slot = torch.where((slot & 1) == 1, pick[slot >> 1], slot)
    return src, src[slot >> 1]


def _chung_lu_edges(n, m, g):
    """Expected degrees ~ power law with exponent 2.3, capped at 800."""
    w = torch.arange(1, n + 1, device=DEV, dtype=torch.float64).pow(-1.0 / 1.3)
    w = torch.clamp(w * (2.0 * m / w.sum()), max=800.0)
    c = torch.cumsum(w, 0)
    def ends():
        return torch.searchsorted(c, torch.rand(m, generator=g, device=DEV, dtype=torch.float64) * c[-1]).clamp(max=n - 1)
    u, v = ends(), ends()
    at = torch.randperm(n, generator=g, device=DEV)  # ids in no order of degree
    return at[u], at[v]


def _edges(kind, n, ef, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    if kind == "ba":
        u, v = _ba_edges(n, max(1, int(ef / 2)), g)
    else:
        u, v = {"rmat": _rmat_edges, "er": _er_edges, "chunglu": _chung_lu_edges}[kind](n, int(n * ef), g)
    return u.to(torch.int32).cpu().numpy(), v.to(torch.int32).cpu().numpy()


# ---------------------------------------------------------------------------
# States

_shared = []


def _context():
    """The one device context a program keeps."""
    if not _shared:
        _shared.append(J.Context(0))
    return _shared[0]


class State:
    """What a program holds between calls; lets its device objects go with itself."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        try:
            for x in ("batch", "server"):
                h = getattr(self, x, None)
                if h is not None:
                    h.free() if x == "batch" else h.stop()
            for G in getattr(self, "graphs", ()):
                G.free()
            own = getattr(self, "own", None)
            if own is not None:
                own.close()
        except Exception:
            pass


def _sub_seed(seed, i):
    return (seed * 1000003 + i * 7919 + 17) & 0x7FFFFFFF


def _many(case, seed, ctx):
    """The case's graphs: sizes log-uniform, half Erdos-Renyi (or all R-MAT for the server)."""
    rng = np.random.default_rng(seed)
    out = []
    for i in range(case["graphs"]):
        n = int(math.exp(rng.uniform(math.log(case["n_min"]), math.log(case["n_max"]))))
        if case["kind"] == "serve":
            kind, ef = "rmat", 16
        elif i % 2 == 0:
            kind, ef = "er", float(rng.uniform(4, 32))
        else:
            kind, ef = "ba", 2 * int(rng.integers(4, 17))
        out.append(ctx.graph_from_edges(n, *_edges(kind, n, ef, _sub_seed(seed, i))))
    return out, rng


def prepare(case, seed):
    gc.collect()
    kind = case["kind"]
    if kind == "query":
        G = _context().graph_from_edges(case["n"], *_edges(case["graph"], case["n"], case["ef"], seed))
        n, k, parts = case["n"], case["part"], case["parts"]
        return State(kind=kind, graphs=[G], patterns=case["patterns"].split(","),
                     roots=None if parts == 1 else (n * k // parts, n * (k + 1) // parts))
    if kind == "edges":
        u, v = _edges(case["graph"], case["n"], case["ef"], seed)
        return State(kind=kind, ctx=_context(), n=case["n"], u=u, v=v, patterns=case["patterns"].split(","))
    if kind == "batch":
        ctx = _context()
        graphs, rng = _many(case, seed, ctx)
        queries = [(G, SMALL_SET[int(rng.integers(0, 4))], 0, None) for G in graphs]
        batch = ctx.prepare_batch(queries) if case["replay"] else None
        return State(kind=kind, ctx=ctx, graphs=graphs, queries=queries, batch=batch)
    ctx = J.Context(0)
    graphs, rng = _many(case, seed, ctx)
    requests = [(graphs[int(rng.integers(0, len(graphs)))], SERVED[int(rng.integers(0, len(SERVED)))])
                for _ in range(case["requests"])]
    return State(kind=kind, own=ctx, graphs=graphs, requests=requests, server=J.Server(ctx))


def run(state):
    if state.kind == "query":
        return [state.graphs[0].count(p, state.roots)[0] for p in state.patterns]
    if state.kind == "edges":
        G = state.ctx.graph_from_edges(state.n, state.u, state.v)
        counts = [G.count(p)[0] for p in state.patterns]
        G.free()
        return counts
    if state.kind == "batch":
        counts, _ = state.batch.run() if state.batch is not None else state.ctx.count_batch(state.queries)
        return np.array(counts, dtype=np.int64)
    tickets = [state.server.submit(G, p) for G, p in state.requests]
    return np.array([state.server.wait(t)[0] for t in tickets], dtype=np.int64)


# ---------------------------------------------------------------------------
# Work and exact values


def _csr_bytes(n, ef):
    return 8.0 * (n + 1) + 4.0 * 2 * n * ef


def work(case):
    """Bytes of the resident symmetric CSR read once per query (counts are a few bytes); an edge
    list is read and its CSR written too.  Duplicate edges are counted, so this is slightly high."""
    if case["kind"] in ("query", "edges"):
        b = _csr_bytes(case["n"], case["ef"]) * len(case["patterns"].split(",")) / case.get("parts", 1)
        if case["kind"] == "edges":
            b += 8.0 * case["n"] * case["ef"] + _csr_bytes(case["n"], case["ef"])
        return {"bytes": b, "flops": 0}
    lo, hi = math.log(case["n_min"]), math.log(case["n_max"])
    mean_n = (case["n_max"] - case["n_min"]) / (hi - lo)
    ef = 16 if case["kind"] == "serve" else 18
    return {"bytes": _csr_bytes(mean_n, ef) * (case["requests"] if case["kind"] == "serve" else case["graphs"]), "flops": 0}


def _dense(case, seed):
    u, v = _edges(case["graph"], case["n"], case["ef"], seed)
    A = torch.zeros(case["n"], case["n"], dtype=torch.float64, device=DEV)
    u, v = torch.from_numpy(u).long().to(DEV), torch.from_numpy(v).long().to(DEV)
    A[u, v] = 1.0
    A[v, u] = 1.0
    A.fill_diagonal_(0.0)
    return A


def _pairs(x):
    return x * (x - 1) / 2


def _exact_one(A, p):
    """Whole-graph counts from dense adjacency products in float64 (all values below 2^53)."""
    n = A.shape[0]
    C = A @ A
    if p == "TC":
        return int((C * A).sum().item()) // 6
    if p == "P2":  # two triangles on an edge
        return int((_pairs(C) * A).sum().item()) // 2
    if p == "P1":  # two common neighbours of a vertex pair
        C.fill_diagonal_(0.0)
        return int(_pairs(C).sum().item()) // 4
    if p == "P4":  # a triangle and a 4-cycle on a common edge, five vertices
        walks = (A @ C) * A  # walks of length 3 between the ends of an edge
        d = A.sum(1)
        t = C * A  # triangles on an edge
        squares = walks - (d[:, None] + d[None, :] - 1) * A  # 4-cycles on the edge
        # for a triangle u v x: the 4-cycles u v y z with x among y, z are t(v,x) - 1 and t(u,x) - 1
        ends = (t @ A) * A
        return int((t * squares - ends - ends.T + 2 * t).sum().item()) // 2
    total = 0
    for x in range(n):  # inside the neighbourhood of each vertex
        nb = A[x].nonzero()[:, 0]
        B = A[nb][:, nb]
        q = B @ B
        if p == "P13":  # triangles
            total += int((q * B).sum().item()) // 6
        else:  # P8: 4-cycles
            q.fill_diagonal_(0.0)
            total += int(_pairs(q).sum().item()) // 4
    return total // 4 if p == "P13" else total


def exact(case, seed):
    if case["kind"] != "query" or case["parts"] != 1 or case["graph"] == "chunglu":
        return None
    patterns = case["patterns"].split(",")
    limit = {"TC": 20000, "P1": 20000, "P2": 20000, "P4": 20000, "P8": 4200, "P13": 4200}
    if any(case["n"] > limit.get(p, 0) for p in patterns):
        return None
    A = _dense(case, seed)
    return [_exact_one(A, p) for p in patterns]
