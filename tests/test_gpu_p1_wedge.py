"""The 4-cycle (P1) kernel at the edges of its root classes: tables at their
wedge limits, counters that pass 16 bits, roots shared by several blocks,
window widths around the dense limit and ids too wide for packed slots.  The
expected counts are closed forms or the wedge identity in numpy (pinned to
the reference nest by test_p1_wedge.py)."""
import numpy as np
import pytest

import jupiter_amd as J

pytestmark = pytest.mark.gpu


def wedge_count(g, rb, re):
    """sum over roots v0 of [rb, re) and x < v0 of C(c_x, 2)."""
    total = 0
    for v0 in range(rb, re):
        low = [v for v in g.col[g.rowptr[v0]:g.rowptr[v0 + 1]] if v < v0]
        if len(low) < 2:
            continue
        x = np.concatenate([g.col[g.rowptr[v]:g.rowptr[v + 1]] for v in low])
        _, c = np.unique(x[x < v0], return_counts=True)
        total += int((c.astype(np.int64) * (c - 1) // 2).sum())
    return total


def bipartite(left, right, nv, hubs_last):
    """Complete bipartite left x right, hubs (the smaller side) at the top or bottom ids of nv."""
    hubs = np.arange(nv - left, nv) if hubs_last else np.arange(left)
    leaves = np.arange(right) if hubs_last else np.arange(nv - right, nv)
    return J.CSR.from_edges(nv, np.repeat(hubs, right), np.tile(leaves, left))


# wedges of the roots at the limits: the hub with rank r over `right` leaves
# has r * right wedges below it (tables of 512 and 1024 wedges, 16-bit counts,
# split roots beyond 2^19 wedges)
@pytest.mark.parametrize("left,right,nv", [
    (2, 3, 5), (3, 511, 600), (3, 512, 600), (2, 1023, 1100), (2, 1024, 1100), (2, 1025, 1100), (5, 4096, 5000),
    (3, 32768, 40000), (2, 65535, 65537), (2, 65536, 70000), (3, 70001, 80000), (9, 65600, 70000)])
@pytest.mark.parametrize("hubs_last", [True, False])
def test_complete_bipartite(ctx, left, right, nv, hubs_last):
    print(f"[case] K_{left},{right} nv {nv} hubs_last {hubs_last}", flush=True)
    G = ctx.upload(bipartite(left, right, nv, hubs_last))
    want = left * (left - 1) // 2 * (right * (right - 1) // 2)
    for _ in range(2):
        assert G.count("P1")[0] == want
    cut = [0, 1, nv // 3, nv - left, nv - 1, nv]
    assert sum(G.count("P1", (a, b))[0] for a, b in zip(cut, cut[1:])) == want
    G.free()


def spread(nv, hubs, deg, seed):
    """Hubs at the top ids, neighbours spread over all ids, plus a sparse random part."""
    rng = np.random.default_rng(seed)
    src = np.repeat(np.arange(nv - hubs, nv), deg)
    dst = rng.integers(0, nv, hubs * deg)
    # half of the neighbours shared by all hubs, so wedges meet
    dst[np.arange(hubs * deg) % 2 == 0] = np.tile(np.sort(rng.integers(0, nv, deg // 2)), hubs)
    more = rng.integers(0, nv, (2, 4 * deg))
    return J.CSR.from_edges(nv, np.concatenate([src, more[0]]), np.concatenate([dst, more[1]]))


# nv around the widths of dense windows (32768 and 2 * that), several windows,
# and beyond 2^22, where more than 1022 neighbours leave packed slots
@pytest.mark.parametrize("nv,hubs,deg", [(32767, 4, 3000), (32769, 4, 3000), (65537, 6, 2000), (300001, 8, 2400),
                                         (4194303, 6, 1100), (5000003, 6, 600), (5000003, 8, 2400)])
def test_windows(ctx, nv, hubs, deg):
    print(f"[case] spread nv {nv} hubs {hubs} deg {deg}", flush=True)
    g = spread(nv, hubs, deg, nv)
    G = ctx.upload(g)
    want = wedge_count(g, 0, nv) if nv < 100000 else wedge_count(g, nv - hubs, nv)
    got = G.count("P1", (0, nv) if nv < 100000 else (nv - hubs, nv))[0]
    assert got == want
    # whole graph (degree order) equals its parts in id order
    parts = [0, nv // 2, nv - hubs, nv - 1, nv]
    assert G.count("P1")[0] == sum(G.count("P1", (a, b))[0] for a, b in zip(parts, parts[1:]))
    G.free()


def test_batch_of_ranges(ctx):
    """Several 4-cycle queries in one launch sequence, ranges and empty ones among them, eager and replayed."""
    gs = [J.rmat(9, 16, seed=4), bipartite(3, 700, 900, True), J.erdos_renyi(777, 9, seed=2), J.rmat(11, 8, seed=5)]
    Gs = [ctx.upload(g) for g in gs]
    q = []
    for g, G in zip(gs, Gs):
        q += [(G, "P1", 0, None), (G, "P1", 5, g.nv // 2), (G, "P1", 7, 7), (G, "P1", g.nv - 1, g.nv)]
    want = [wedge_count(g, a, b) for g in gs for a, b in ((0, g.nv), (5, g.nv // 2), (7, 7), (g.nv - 1, g.nv))]
    assert ctx.count_batch(q)[0] == want
    with ctx.prepare_batch(q) as B:
        for _ in range(3):
            assert B.run()[0] == want
            assert Gs[0].count("P1")[0] == want[0]
    for G in Gs:
        G.free()
