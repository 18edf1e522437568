"""The triangle sums (P5, P7, P9, P11, P12) and per-edge triangle counts at
the edges of their tiers: roots of 63 to 66 neighbours, rows in the small and
the large LDS tier and in global memory, hubs and non-hubs, vertex counts
around the bitmap's word, root ranges of both routes.  Bar: bit-exact against
the oracle, or against the per-edge kernels over small root ranges (held to
the oracle in test_gpu_sym.py) where the oracle would take minutes."""
import itertools
from math import comb

import numpy as np
import pytest

import jupiter_amd as J
import oracle_lib as O

pytestmark = pytest.mark.gpu
PATS = ["P2", "P5", "P7", "P9", "P11", "P12"]


def complete(n, extra=0):
    e = np.array(list(itertools.combinations(range(n), 2)), dtype=np.int32)
    return J.CSR.from_edges(n + extra, e[:, 0], e[:, 1])


def core_and_leaves(core, leaves, per_leaf, seed):
    """A random core (half its pairs joined) and leaves joined to per_leaf core vertices each; ids shuffled."""
    rng = np.random.default_rng(seed)
    pairs = np.array(list(itertools.combinations(range(core), 2)))
    pairs = pairs[rng.random(len(pairs)) < 0.5]
    src = np.repeat(np.arange(core, core + leaves), per_leaf)
    dst = rng.integers(0, core, leaves * per_leaf)
    perm = rng.permutation(core + leaves)
    return J.CSR.from_edges(core + leaves, perm[np.concatenate([pairs[:, 0], src])],
                            perm[np.concatenate([pairs[:, 1], dst])])


# vertices of each pattern: K_n holds C(n, k) / C(7, k) times what K_7 holds
SIZE = {"P2": 4, "P5": 5, "P7": 5, "P9": 5, "P11": 6, "P12": 6}


@pytest.mark.parametrize("n,extra", [(3, 0), (5, 27), (33, 0), (63, 1), (64, 0), (65, 0), (66, 70), (130, 0), (200, 3)])
def test_complete_graphs(ctx, n, extra):
    """K_n: roots of every degree up to n - 1 in one wave, then in a block."""
    k7 = complete(7)
    G = ctx.upload(complete(n, extra))
    for p in PATS:
        print(f"[case] K{n}+{extra} {p}", flush=True)
        want = O.count(k7.rowptr, k7.col, J.PATTERNS[p]) * comb(n, SIZE[p]) // comb(7, SIZE[p])
        assert G.count(p)[0] == want, p
        cut = [0, n // 3, n // 2, n + extra]
        assert sum(G.count(p, (a, b))[0] for a, b in zip(cut, cut[1:])) == want, p
    G.free()


@pytest.mark.parametrize("g", [lambda: core_and_leaves(40, 500, 5, 1), lambda: core_and_leaves(70, 800, 6, 2),
                               lambda: J.rmat(9, 12, seed=11), lambda: J.erdos_renyi(1023, 20, seed=3)])
def test_ranges_against_oracle(ctx, g):
    g = g()
    G = ctx.upload(g)
    n = g.nv
    for p in PATS:
        print(f"[case] nv {n} {p}", flush=True)
        for a, b in ((0, n), (0, n // 2), (n // 2, n), (n // 5, n - 7), (n - 3, n)):
            assert G.count(p, (a, b))[0] == O.count(g.rowptr, g.col, J.PATTERNS[p], a, b), (p, a, b)
    G.free()


@pytest.mark.parametrize("core,leaves,per_leaf", [(60, 3000, 12), (150, 60000, 20), (170, 120000, 22)])
def test_wide_rows(ctx, core, leaves, per_leaf):
    """Rows beyond the small LDS tier and beyond LDS: the whole graph (triangle sums) equals the sum of
    root ranges each too small for that route (per-edge kernels)."""
    g = core_and_leaves(core, leaves, per_leaf, core + leaves)
    G = ctx.upload(g)
    ends = np.searchsorted(g.rowptr, np.arange(65) * g.nnz // 64)
    # a core vertex holds a large share of the edges: alone in its range
    hubs = np.nonzero(g.degrees() > g.nnz // 256)[0]
    cut = sorted(set(ends.tolist()) | set(hubs.tolist()) | set((hubs + 1).tolist()) | {0, g.nv})
    share = max(int(g.rowptr[b] - g.rowptr[a]) for a, b in zip(cut, cut[1:]))
    assert share < g.nnz // 32
    for p in PATS:
        print(f"[case] core {core} leaves {leaves} {p}", flush=True)
        assert G.count(p)[0] == sum(G.count(p, (a, b))[0] for a, b in zip(cut, cut[1:])), p
    G.free()
