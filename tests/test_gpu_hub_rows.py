"""Cliques with the rows of the last places of the DAG's order read from
bitmaps: closed forms on complete graphs around the tiers and the bitmaps'
lines, and every tier against the general path of the no-allocation entry
point, on graphs with members outside the bitmaps, on DAGs in another order
than the degrees', and on root ranges."""
from math import comb

import numpy as np
import pytest

import jupiter_amd as J
from test_zz_no_alloc import complete, noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [183, 258, 514, 1026, 1060])
def test_complete(ctx, n):
    G = ctx.upload(complete(n))
    for p, k in (("TC", 3), ("P13", 4)) + ((("P14", 5),) if n <= 514 else ()):
        print(f"[case] K{n} {p}", flush=True)
        assert G.count(p)[0] == comb(n, k), p
        assert G.count(p, (n // 2, n))[0] == noalloc(G, p, (n // 2, n)), p
    G.free()


def reordered(g, seed):
    """The graph's edges directed along a random order of the vertices."""
    rank = np.random.default_rng(seed).permutation(g.nv)
    src = np.repeat(np.arange(g.nv), np.diff(g.rowptr))
    keep = rank[src] < rank[g.col]
    rp = np.zeros(g.nv + 1, np.int64)
    np.cumsum(np.bincount(src[keep], minlength=g.nv), out=rp[1:])
    return J.CSR(rp, g.col[keep])


GRAPHS = {
    "rmat13": lambda: (J.rmat(13, 16, seed=2), J.SYM),
    "rmat16": lambda: (J.rmat(16, 16, seed=2), J.SYM),  # 65,536 vertices, 16,384 rows
    "sparse": lambda: (J.erdos_renyi(60000, 3.0, seed=3), J.SYM),
    "dense": lambda: (J.erdos_renyi(900, 500.0, seed=4), J.SYM),
    "dag13": lambda: (reordered(J.rmat(13, 16, seed=2), 5), J.DAG),
    "dag16": lambda: (reordered(J.rmat(15, 16, seed=3), 6), J.DAG),
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_against_general_path(ctx, name):
    g, flags = GRAPHS[name]()
    G = ctx.upload(g, flags)
    n = g.nv
    for p in ("TC", "P13", "P14") + (("P15",) if name in ("dense", "rmat13", "sparse") else ()):
        for r in (None, (0, n // 3), (n // 3, n)):
            print(f"[case] {name} {p} {r}", flush=True)
            assert G.count(p, r)[0] == noalloc(G, p, r), (name, p, r)
    G.free()


@pytest.mark.parametrize("copies", [1, 300])
def test_small_roots(ctx, copies):
    """Disjoint cliques of 2 to 36 vertices, without bitmaps and with some of
    the members outside them: roots of 1 to 35 members, batched and not."""
    u, v, n = [], [], 0
    sizes = list(range(2, 37))
    for s in sizes:
        a, b = np.triu_indices(s, 1)
        u.append(n + a)
        v.append(n + b)
        n += s
    u, v = np.concatenate(u), np.concatenate(v)
    shift = np.repeat(np.arange(copies) * n, len(u))
    perm = np.random.default_rng(1).permutation(n * copies) if copies > 1 else np.arange(n)
    g = J.CSR.from_edges(n * copies, perm[np.tile(u, copies) + shift], perm[np.tile(v, copies) + shift])
    G = ctx.upload(g)
    for p, k in (("TC", 3), ("P13", 4), ("P14", 5)):
        print(f"[case] cliques x {copies} {p}", flush=True)
        assert G.count(p)[0] == copies * sum(comb(s, k) for s in sizes), p
    G.free()
