"""GPU: the one-launch peel gives up its waits and the host peels in steps; the limits are set from the host, every
block of the launch leaves by itself.  Entry for entry against the oracle."""
import numpy as np
import pytest

import kcgpu_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# at the first wait, and at the second (degrees half decremented, some priorities written, the first frontier gone)
@pytest.mark.parametrize("wait", ["0", "100000,0"])
@pytest.mark.parametrize("n,m,hub", [(200, 900, 40), (1500, 9000, 300), (40_000, 260_000, 800), (120_000, 800_000, 30_000)])
def test_peel_gives_up_and_is_stepped(n, m, hub, wait, monkeypatch):
    G = K.Graph.generate(K.GEN_CHUNG_LU, seed=n, n=n, m=m, gamma=2.1, max_degree=hub)
    rp, col = G.csr()
    rp = rp.astype(np.uint64)
    prio, core = O.peel_priority(rp, col)
    erp, ec = O.orient(rp, col, prio)
    monkeypatch.setenv("KC_PEEL_WAIT_US", wait)
    for _ in range(2):
        o = G.orient("degen")
        orp, oc, key = o.export()
        assert (key == prio).all() and o.info()["max_core"] == core
        assert (orp == erp).all() and (oc == ec).all()
        o.close()
    monkeypatch.delenv("KC_PEEL_WAIT_US")
    o = G.orient("degen")  # the waits hold again, on the same device blocks
    assert (o.export()[2] == prio).all() and o.info()["max_core"] == core


# where the peel's lists and hub queues lie: the smallest graphs, and hubs at both sides of the room for their queues
@pytest.mark.parametrize("n,hubs", [(1, 0), (2, 1), (3, 1), (4, 2), (5, 3), (9000, 1), (4200, 4200), (6500, 900)])
def test_peel_of_smallest_and_hub_graphs(n, hubs):
    """`hubs` vertices joined to every other vertex: with 4,200 of 4,200 the rows of all are above 4,096 entries"""
    if hubs == n:
        a, b = np.triu_indices(n, 1)
    else:
        a = np.repeat(np.arange(hubs), n)
        b = np.tile(np.arange(n), hubs)
        keep = a < b
        a, b = a[keep], b[keep]
    G = K.Graph.from_edges(a.astype(np.uint32), b.astype(np.uint32), n)
    o = G.orient("degen")
    rp, col, key = o.export()
    if hubs < n or n == 1:
        prio, core = O.peel_priority(G.csr()[0].astype(np.uint64), G.csr()[1])
        assert (key == prio).all() and o.info()["max_core"] == core
    else:  # a clique goes in one round at level n - 1, which empties the graph and assigns nothing
        assert int(rp[-1]) == a.size and o.info()["max_core"] == n - 1 and (key == 2 * a.size).all()
