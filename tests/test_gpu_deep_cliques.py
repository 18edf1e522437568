"""P14, P15 and P16 where their sets cross a word or a class: complete
graphs with roots and sets of 24/25, 63 to 66, 127 to 130 and 255 to 258
members (closed forms), and dense random graphs against the oracle and
against the fused kernels of the no-allocation entry point."""
from math import comb

import numpy as np
import pytest

import jupiter_amd as J
import oracle_lib as O
from test_zz_no_alloc import complete, noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 6, 7, 25, 26, 27, 64, 65, 66, 67, 68, 128, 129, 130, 131, 132])
def test_complete(ctx, n):
    G = ctx.upload(complete(n))
    for p, k in (("P14", 5), ("P15", 6), ("P16", 7)):
        print(f"[case] K{n} {p}", flush=True)
        assert G.count(p)[0] == comb(n, k), p
    G.free()


@pytest.mark.parametrize("n", [194, 257, 259, 262])
def test_complete_wide(ctx, n):
    G = ctx.upload(complete(n))
    for p, k in (("P14", 5), ("P15", 6)):
        print(f"[case] K{n} {p}", flush=True)
        assert G.count(p)[0] == comb(n, k), p
    G.free()


def dense(n, p, seed):
    rng = np.random.default_rng(seed)
    u, v = np.triu_indices(n, 1)
    keep = rng.random(len(u)) < p
    perm = rng.permutation(n)
    return J.CSR.from_edges(n, perm[u[keep]], perm[v[keep]])


@pytest.mark.parametrize("n,p,pats", [(40, 0.8, ("P14", "P15", "P16")), (90, 0.6, ("P14", "P15", "P16")),
                                      (180, 0.5, ("P14", "P15", "P16")), (400, 0.35, ("P14", "P15")),
                                      (700, 0.3, ("P15",))])
def test_dense_random(ctx, n, p, pats):
    g = dense(n, p, n)
    d = g.orient()
    G = ctx.upload(g)
    for name in pats:
        print(f"[case] G({n},{p}) {name}", flush=True)
        got = G.count(name)[0]
        assert got == noalloc(G, name), name
        if n <= 180:
            assert got == O.count(d.rowptr, d.col, J.PATTERNS[name]), name
        half = n // 2
        assert G.count(name, (0, half))[0] + G.count(name, (half, n))[0] == got, name
    G.free()
