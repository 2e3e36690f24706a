"""GPU: the degeneracy peel against the oracle, entry for entry, on the shapes that take its different ways."""
import numpy as np
import pytest

import kcgpu_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _edges(shape):
    r = np.random.default_rng(7)
    if shape == "path":  # one long chain of rounds at level 1
        a = np.arange(4999)
        return a, a + 1, 5000
    if shape == "star":  # a hub row above 4,096 entries, emptied in two rounds
        return np.zeros(9000, int), np.arange(1, 9001), 9001
    if shape == "cliques":  # levels far apart, empty ones skipped
        e = [np.triu_indices(s, 1) for s in (3, 40, 90, 200)]
        off = [0, 3, 43, 133]
        return np.concatenate([o + a for o, (a, _) in zip(off, e)]), np.concatenate([o + b for o, (_, b) in zip(off, e)]), 340
    if shape == "isolated":  # level 0, and a last round that is assigned nothing
        return np.array([3]), np.array([700]), 2000
    if shape == "rows64":  # rows of 63, 64, 65 and 66 entries
        src, dst, at = [], [], 0
        for d in (63, 64, 65, 66):
            src.append(np.full(d, at))
            dst.append(at + 1 + np.arange(d))
            at += d + 1
        return np.concatenate(src), np.concatenate(dst), at
    if shape == "dense_core":  # hubs above 4,096 inside a core, long tails of short rows
        a = r.integers(0, 12, 60_000)
        b = r.integers(0, 20_000, 60_000)
        x, y = np.triu_indices(300, 1)
        return np.concatenate([a, x]), np.concatenate([b, y]), 20_000
    raise ValueError(shape)


@pytest.mark.parametrize("shape", ["path", "star", "cliques", "isolated", "rows64", "dense_core"])
@pytest.mark.parametrize("mode", ["", "step"])
def test_peel_shapes_vs_oracle(shape, mode, monkeypatch):
    if mode:
        monkeypatch.setenv("KC_PEEL_MODE", mode)
    s, d, n = _edges(shape)
    G = K.Graph.from_edges(s.astype(np.uint32), d.astype(np.uint32), n)
    rp, col = G.csr()
    rp = rp.astype(np.uint64)
    prio, core = O.peel_priority(rp, col)
    o = G.orient("degen")
    orp, oc, key = o.export()
    assert (key == prio).all() and o.info()["max_core"] == core
    erp, ec = O.orient(rp, col, prio)
    assert (orp == erp).all() and (oc == ec).all()


@pytest.mark.parametrize("n,m,hub", [(1500, 9000, 300), (40_000, 260_000, 800), (300_000, 1_900_000, 6000)])
def test_peel_power_law_vs_oracle(n, m, hub):
    G = K.Graph.generate(K.GEN_CHUNG_LU, seed=n, n=n, m=m, gamma=2.1, max_degree=hub)
    rp, col = G.csr()
    prio, core = O.peel_priority(rp.astype(np.uint64), col)
    for _ in range(3):
        o = G.orient("degen")
        assert (o.export()[2] == prio).all() and o.info()["max_core"] == core
