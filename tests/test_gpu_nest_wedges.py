"""P4, P6, P8 and P10 as wedge counts (on the graph, or on the induced
neighbourhoods): root ranges of every size, slivers (which run per edge) among
them, graphs with more vertices than a dense counter window, hubs whose
tasks are windows, complete graphs.  Bar: bit-exact against the oracle."""
import itertools

import numpy as np
import pytest

import jupiter_amd as J
import oracle_lib as O

pytestmark = pytest.mark.gpu
PATS = ["P4", "P6", "P8", "P10"]


def planted(nv, mean_degree, cliques, size, seed):
    """A sparse random graph with cliques planted among all ids."""
    rng = np.random.default_rng(seed)
    m = int(nv * mean_degree / 2)
    u, v = rng.integers(0, nv, (2, m))
    for _ in range(cliques):
        c = rng.choice(nv, size, replace=False)
        e = np.array(list(itertools.combinations(c, 2)))
        u, v = np.concatenate([u, e[:, 0]]), np.concatenate([v, e[:, 1]])
    return J.CSR.from_edges(nv, u, v)


def wheel(rim, hubs, seed):
    """hubs vertices joined to all of a cycle with chords: wide neighbourhoods, ids shuffled."""
    rng = np.random.default_rng(seed)
    n = rim + hubs
    r = np.arange(rim)
    u = np.concatenate([r, r, np.repeat(np.arange(rim, n), rim)])
    v = np.concatenate([(r + 1) % rim, (r + 2) % rim, np.tile(r, hubs)])
    perm = rng.permutation(n)
    return J.CSR.from_edges(n, perm[u], perm[v])


CASES = {
    "er": lambda: J.erdos_renyi(600, 14, seed=3), "rmat": lambda: J.rmat(7, 14, seed=5),
    "planted_small": lambda: planted(500, 4, 6, 14, 1), "planted_32768": lambda: planted(32768, 6, 30, 9, 2),
    "planted_70001": lambda: planted(70001, 6, 40, 9, 3), "wheel_1_hub": lambda: wheel(900, 1, 4),
    "wheel_3_hubs": lambda: wheel(300, 3, 5), "k30": lambda: planted(30, 1, 1, 30, 6),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_against_oracle(ctx, name):
    g = CASES[name]()
    G = ctx.upload(g)
    n = g.nv
    hub = int(np.argmax(g.degrees()))
    for p in PATS:
        for a, b in ((0, n), (0, n // 2), (n // 2, n), (n // 7, n - 5), (hub, hub + 1), (n - 2, n), (3, 3)):
            print(f"[case] {name} {p} [{a}, {b})", flush=True)
            assert G.count(p, (a, b))[0] == O.count(g.rowptr, g.col, J.PATTERNS[p], a, b), (p, a, b)
    G.free()


def test_wide_windows(ctx):
    """Neighbourhoods and lists wider than a block's counters: whole graphs equal the sum of their parts,
    and P8 the closed form (4-cycles of the rim inside each hub's neighbourhood and through hub pairs)."""
    rim, hubs = 70000, 2
    g = wheel(rim, hubs, 9)
    G = ctx.upload(g)
    n = g.nv
    cut = [0, 1, n // 3, n // 2, n - 1, n]
    for p in PATS:
        print(f"[case] wheel {rim}+{hubs} {p}", flush=True)
        whole = G.count(p)[0]
        assert whole == sum(G.count(p, (a, b))[0] for a, b in zip(cut, cut[1:])), p
        if p == "P8":
            # the square of a cycle has per rim vertex i the 4-cycles i, i+1, i+2, i+3 (by i-i+1-i+3-i+2) and
            # no other; every hub sees the whole rim; a rim vertex sees its 4 rim neighbours and both hubs
            around = O_rim_vertex()
            assert whole == hubs * rim + rim * around
    G.free()


def O_rim_vertex():
    """4-cycles in the neighbourhood of one rim vertex (4 rim neighbours, 2 hubs joined to them), brute force."""
    v = [-2, -1, 1, 2, "a", "b"]
    adj = {(x, y) for x in v for y in v if x != y and
           (isinstance(x, str) != isinstance(y, str) or (not isinstance(x, str) and abs(x - y) <= 2))}
    c = sum(1 for q in itertools.permutations(v, 4)
            if (q[0], q[1]) in adj and (q[1], q[2]) in adj and (q[2], q[3]) in adj and (q[3], q[0]) in adj)
    return c // 8
