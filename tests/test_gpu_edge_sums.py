"""P3, tailed triangles and 3-stars as sums over a root range's edges: exact
against the oracle on whole graphs, on ranges whose twice-the-value partial
sums are odd, and on graphs without triangles."""
import numpy as np
import pytest

import jupiter_amd as J
import oracle_lib as O

pytestmark = pytest.mark.gpu


def clique(n):
    u, v = np.triu_indices(n, 1)
    return J.CSR.from_edges(n, u, v)


GRAPHS = {
    "rmat10": lambda: J.rmat(10, 16, seed=3),
    "ba": lambda: J.barabasi_albert(2000, 6, seed=5),
    "sparse": lambda: J.erdos_renyi(700, 3.0, seed=2),
    "k33": lambda: clique(33),
    "star": lambda: J.CSR.from_edges(300, np.zeros(299, np.int32), np.arange(1, 300)),
}


@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_edge_sums_match_oracle(ctx, name):
    g = GRAPHS[name]()
    G = ctx.upload(g)
    n = g.nv
    for a, b in [(0, n), (0, 1), (n // 3, n // 2), (n - 7, n), (n // 2, n // 2)]:
        r = None if (a, b) == (0, n) else (a, b)
        assert G.count("P3", r)[0] == O.count(g.rowptr, g.col, 3, a, b), (name, a, b)
        assert G.count("TAILTRI", r)[0] == O.vertex_sums(g.rowptr, g.col, 1, a, b), (name, a, b)
        assert G.count("STAR3", r)[0] == O.vertex_sums(g.rowptr, g.col, 0, a, b), (name, a, b)
    G.free()


def test_served_without_room_for_workspaces(ctx):
    """A budget that admits the requests but leaves their lanes little room
    (32 MiB: induced neighbourhoods in parts; 4 MiB: bitmaps for few hubs or
    none) for the optional workspaces: same counts."""
    G = ctx.upload(J.rmat(11, 16, seed=3))
    pats = ["P4", "P5", "P6", "P8", "P9", "P10", "P15", "P3"]
    alone = [G.count(p)[0] for p in pats]
    for mib in (512, 64):
        with J.Server(ctx, hbm_budget_bytes=mib << 20, heavy_lanes=16) as srv:
            tickets = [srv.submit(G, p) for p in pats]
            assert [srv.wait(t)[0] for t in tickets] == alone
    G.free()
