"""Clique roots of few members on uploaded DAGs whose hubs come early in the
order: a member's list may be long (searched for the root's members) or not
(streamed), at every ratio between the two; single queries and batches.  Bar:
the oracle, and a closed form where the lists of one wave's roots together
pass 2^31 elements."""
import numpy as np
import pytest

import jupiter_amd as J
import oracle_lib as O

pytestmark = pytest.mark.gpu
PATS = ["TC", "P13", "P14"]


def early_hubs(small, hubs, targets, seed):
    """Edges point to larger ids: small roots (up to 32 members) -> hubs of 64 to 1,800 out-neighbours -> targets."""
    rng = np.random.default_rng(seed)
    h0, t0 = small, small + hubs
    nv = t0 + targets
    src, dst = [], []
    for v in range(small):
        d = int(rng.integers(2, 33))
        m = rng.choice(np.arange(h0, nv), d, replace=False)
        k = int(rng.integers(0, min(d, hubs) + 1))
        m = np.unique(np.concatenate([rng.choice(np.arange(h0, t0), k, replace=False), m]))[:32]
        src.append(np.full(len(m), v))
        dst.append(m)
    for i in range(hubs):
        d = [64, 65, 66, 256, 257, 1800][i % 6]
        m = rng.choice(np.arange(h0 + i + 1, nv), d, replace=False)
        src.append(np.full(d, h0 + i))
        dst.append(m)
    a, b = rng.integers(t0, nv, 30000), rng.integers(t0, nv, 30000)
    src.append(np.minimum(a, b)[a != b])
    dst.append(np.maximum(a, b)[a != b])
    key = np.unique(np.concatenate(src).astype(np.int64) * nv + np.concatenate(dst))
    s, c = key // nv, (key % nv).astype(np.int32)
    rp = np.zeros(nv + 1, np.int64)
    np.cumsum(np.bincount(s, minlength=nv), out=rp[1:])
    return J.CSR(rp, c)


@pytest.mark.parametrize("small,hubs,targets", [(500, 12, 2000), (64, 40, 2200), (3000, 24, 1900)])
def test_members_with_long_lists(ctx, small, hubs, targets):
    g = early_hubs(small, hubs, targets, small)
    want = {p: O.count(g.rowptr, g.col, J.PATTERNS[p]) for p in PATS}
    part = {p: O.count(g.rowptr, g.col, J.PATTERNS[p], 0, small) for p in PATS}
    assert want["P14"] > 0 and part["P14"] > 0
    G = ctx.upload(g, flags=J.DAG)
    try:
        for ratio in (1, 8, 32, 1 << 20):
            ctx.set_tuning(gallop_ratio=ratio)
            for p in PATS:
                print(f"[case] {small} roots, {hubs} hubs, ratio {ratio}, {p}", flush=True)
                assert G.count(p)[0] == want[p], (ratio, p)
                assert G.count(p, (0, small))[0] == part[p], (ratio, p)
            got, _ = ctx.count_batch([(G, p, 0, end) for p in PATS for end in (None, small)])
            assert list(got) == [x[p] for p in PATS for x in (want, part)], ratio
    finally:
        ctx.set_tuning(gallop_ratio=-1)
    G.free()


def test_lists_of_a_batch_pass_31_bits(ctx):
    """64 roots of two members, each the same vertex with 34 million out-neighbours and one of those: one triangle a root."""
    n, small = 34_000_000, 64
    h = small
    rp = np.concatenate([np.arange(0, 2 * small + 1, 2), np.full(n + 1, 2 * small + n)]).astype(np.int64)
    col = np.empty(2 * small + n, np.int32)
    col[0:2 * small:2] = h
    col[1:2 * small:2] = h + 1 + np.arange(small) * 500_000
    col[2 * small:] = np.arange(h + 1, h + 1 + n)
    assert small * n > 1 << 31
    print("[case] 64 roots on a list of 34 million", flush=True)
    G = ctx.upload(J.CSR(rp, col), flags=J.DAG)
    assert G.count("TC", (0, small))[0] == small
    got, _ = ctx.count_batch([(G, "TC", 0, small)])
    assert list(got) == [small]
    G.free()
