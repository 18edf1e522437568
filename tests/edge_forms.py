"""Counts of P5, P7, P9, P11 and P12 over a root range, edge by edge with Python sets: for an edge (v0, v1) of
the range, S = N(v0) & N(v1), q(v2) = |S & N(v2)| and t the common neighbours of an edge.  Held to the oracle by
test_edge_forms.py; for graphs on which the oracle's nests take minutes."""


def pairs(x):
    return x * (x - 1) // 2


def counts(g, rb, re, plant=False):
    """{pattern: count} over the roots [rb, re); plant adds the edge's own ends to every q."""
    rp, ci = g.rowptr, g.col
    nbr = {}

    def n(v):
        if v not in nbr:
            nbr[v] = set(ci[rp[v]:rp[v + 1]].tolist())
        return nbr[v]

    tot = dict.fromkeys(("P5", "P7", "P9", "P11", "P12"), 0)
    for v0 in range(rb, re):
        t0 = {v2: len(n(v0) & n(v2)) for v2 in n(v0)}
        for v1 in n(v0):
            S = n(v0) & n(v1)
            s = len(S)
            if s == 0:
                continue
            q = {v2: len(S & n(v2)) + plant for v2 in S}
            if v1 < v0:
                tot["P5"] += (s - 2) * sum(q.values()) // 2
            else:
                tot["P12"] += (s - 3) * sum(pairs(x) for x in q.values())
            for v2 in S:
                if v2 <= v1:
                    continue
                b = t0[v2] - 1
                tot["P7"] += (s - 1) * b - q[v2]
                if v1 > v0:
                    c = len(n(v1) & n(v2)) - 1
                    tot["P9"] += pairs(q[v2])
                    tot["P11"] += (s - 1) * b * c - q[v2] * (s - 1 + b + c) + 2 * q[v2]
    return tot
