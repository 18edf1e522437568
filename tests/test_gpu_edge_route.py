"""The per-edge launches of P5, P7, P9, P11 and P12 at every shape of the
heavy-edge kernel, over the two hubs of a graph whose other edges make the
pass over all triangles the longer way: edges of 1,200 to 8,193 common
neighbours (the narrow and the 8,192-wide shape, the one with the list in
scratch), S as a vertex bitmap (up to 2^18 vertices), in a hash (beyond), and
graphs beyond 2^20 vertices, where the widest edges run in a wave.  The
profile's kernel names show the route.  Bar: the edge-by-edge forms that
test_edge_forms.py holds to the oracle, bit-exact."""
import numpy as np
import pytest

import edge_forms
import jupiter_amd as J

pytestmark = pytest.mark.gpu


def two_hubs(m, nv, seed):
    """Vertices 0 and 1 joined to each other and to m common neighbours with 40,000 random edges among them; the
    other vertices are a random graph of mean degree 24."""
    rng = np.random.default_rng(seed)
    com = np.arange(2, m + 2)
    a, b = rng.integers(2, m + 2, (2, 40000))
    rest = nv - m - 2
    x, y = rng.integers(m + 2, nv, (2, 12 * rest))
    src = np.concatenate([[0], np.zeros(m, np.int64), np.ones(m, np.int64), a, x])
    dst = np.concatenate([[1], com, com, b, y])
    keep = src != dst
    return J.CSR.from_edges(nv, src[keep], dst[keep])


@pytest.mark.parametrize("m,nv", [(1200, 250_000), (1200, 400_000), (8192, 250_000), (8193, 250_000), (8192, 400_000),
                                  (8193, 400_000), (8193, 1_100_000)])
def test_heavy_shapes(ctx, m, nv):
    g = two_hubs(m, nv, m + nv)
    assert len(np.intersect1d(g.col[g.rowptr[0]:g.rowptr[1]], g.col[g.rowptr[1]:g.rowptr[2]])) == m
    want = edge_forms.counts(g, 0, 2)
    assert min(want.values()) > 0
    G = ctx.upload(g)
    try:
        for h in (1, 32, 1000, 8192):
            ctx.set_tuning(sym_heavy_min=h)
            for p, w in want.items():
                print(f"[case] {m} common, nv {nv}, heavy_min {h}, {p}", flush=True)
                assert G.count(p, (0, 2))[0] == w, (h, p)
                names = {n for n, _ in ctx.last_profile()}
                assert f"sym_{p.lower()}_tri" not in names, (h, p)
                assert (f"sym_{p.lower()}_heavy" in names) == (h < 8192), (h, p)
    finally:
        ctx.set_tuning(sym_heavy_min=-1)
    G.free()
