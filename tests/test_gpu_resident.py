"""GPU: the serving loop's resident launch at the sizes where its tree walk changes words (32 and 64 vertices)."""
import time

import numpy as np
import pytest

import kcgpu_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("density", [0.45, 0.85, 1.0])
def test_resident_launch_at_word_edges(density):
    """graphs whose largest task has 31..34 and 62..64 vertices, k = 3..9, against the oracle"""
    srv = K.Server(workers=1)
    try:
        graphs, want = [], {}
        for n in (32, 33, 34, 35, 63, 64, 65):
            r = np.random.default_rng(n)
            a, b = np.triu_indices(n, 1)
            keep = (r.random(a.size) < density) | (a == 0)
            src = np.concatenate([a[keep], [0, 1]]).astype(np.uint32)
            dst = np.concatenate([b[keep], [n, n]]).astype(np.uint32)  # (vertex n: a second, tiny task)
            G = K.Graph.from_edges(src, dst, n + 1)
            rp, col = G.csr()
            orp, oc = O.orient(rp.astype(np.uint64), col)
            graphs.append((n, srv.add_graph(G, "degree"), orp, oc))
        for n, gid, orp, oc in graphs:  # (all resident first: a running launch does not see a graph added since)
            for k in range(3, 10):
                exp = O.count(orp, oc, k, "pivot_tails", "node")["count"]
                for gran in ("node", "edge"):
                    want[srv.submit(gid, k, "pivot", gran)] = (exp, n, k, gran)
        asked, t0 = len(want), time.perf_counter()
        while want and time.perf_counter() - t0 < 60.0:
            for t in list(want):
                res = srv.poll(t)
                if res is not None:
                    exp, n, k, gran = want.pop(t)
                    assert res.count == exp, (n, k, gran)
            time.sleep(0.0005)
        assert not want
        assert srv.stats()["resident_admitted"] == asked  # none went to a worker
    finally:
        srv.close()
