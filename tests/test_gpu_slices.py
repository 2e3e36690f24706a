"""GPU: counts whose large size classes share the HBM slices of one scratch block."""
import time
from math import comb

import numpy as np
import pytest

import kcgpu_amd as K

pytestmark = pytest.mark.gpu


def _pairs_graph(parts):
    """all edges between `parts` pairs of vertices but none inside a pair: C(parts, k) * 2^k k-cliques.
    Degrees are equal, so out-lists are the later ids: sizes 0..2 * parts - 2, each about once."""
    a, b = np.triu_indices(2 * parts, 1)
    keep = a // 2 != b // 2
    return K.Graph.from_edges(a[keep].astype(np.uint32), b[keep].astype(np.uint32), 2 * parts)


def _cliques(parts, k):
    return comb(parts, k) << k


# 34 tasks above 1024 vertices, whose launch is first, and 512 of 513..1024, whose slices together are larger
PARTS = 530


def test_slices_of_both_hbm_classes():
    G = _pairs_graph(PARTS)
    for k in (3, 4, 5):
        o = G.orient("degree")  # (a new handle: its scratch holds nothing yet)
        assert o.info()["max_out_degree"] == 2 * PARTS - 2
        for _ in range(2):
            r = o.count(k, "pivot", "node", part_size=1)
            assert r.count == _cliques(PARTS, k), k
            assert r.raw["class_tasks"][5] == 2 * (PARTS - 1) - 1024 and r.raw["class_tasks"][4] == 512, k
        assert o.count_noalloc(k, "pivot", "node").count == _cliques(PARTS, k), k
        print("k", k, "done", flush=True)
        o.close()


def test_two_workers_grow_their_slices_side_by_side():
    """Both workers' scratch grows while the other counts and graphs are oriented on the library's stream."""
    graphs = {p: _pairs_graph(p) for p in (PARTS, PARTS + 2, 270)}
    small = K.Graph.generate(K.GEN_BA, seed=7, n=20000, attach=8)
    ref = small.orient("degen").count(5, "pivot", "node").count
    srv = K.Server(workers=2, max_batch=1)
    try:
        gid = {p: srv.add_graph(G, "degree") for p, G in graphs.items()}
        want = {}
        for k in (3, 4, 5, 4):
            for p in graphs:
                want[srv.submit(gid[p], k, "pivot", "node")] = (_cliques(p, k), p, k)
        t0 = time.perf_counter()
        while want and time.perf_counter() - t0 < 60.0:
            o = small.orient("degen")
            assert o.count(5, "pivot", "node").count == ref
            o.close()
            for t in list(want):
                r = srv.poll(t)
                if r is not None:
                    exp, p, k = want.pop(t)
                    assert r.count == exp, (p, k)
                    print("parts", p, "k", k, f"{time.perf_counter() - t0:.2f} s", flush=True)
        assert not want
    finally:
        srv.close()
