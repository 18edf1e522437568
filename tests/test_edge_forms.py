"""The edge-by-edge forms of tests/edge_forms.py equal the oracle over root ranges, and a planted mistake does not."""
import pytest

import edge_forms
import jupiter_amd as J
import oracle_lib as O


@pytest.mark.parametrize("g", [lambda: J.rmat(7, 10, seed=2), lambda: J.erdos_renyi(90, 20, seed=4),
                               lambda: J.barabasi_albert(150, 7, seed=5)])
def test_forms_equal_oracle(g):
    g = g()
    n = g.nv
    for a, b in ((0, n), (0, n // 3), (n // 2, n - 2)):
        got = edge_forms.counts(g, a, b)
        bad = edge_forms.counts(g, a, b, plant=True)
        for p, x in got.items():
            assert x == O.count(g.rowptr, g.col, J.PATTERNS[p], a, b), (p, a, b)
            assert (a, b) != (0, n) or bad[p] != x, p
