"""GPU: pivoting at the line between the register kernels without and with matrix operands (five vertices below a
task's root: k = 7 for edge tasks, 6 for node tasks), alone and with both sides of it in one launch."""
import numpy as np
import pytest

import kcgpu_amd as K
from oracle import oracle as O
from test_gpu_errors import write_oriented

pytestmark = pytest.mark.gpu


def _dense(n, density, seed):
    r = np.random.default_rng(seed)
    a, b = np.triu_indices(n, 1)
    keep = r.random(a.size) < density
    return K.Graph.from_edges(a[keep].astype(np.uint32), b[keep].astype(np.uint32), n)


@pytest.mark.parametrize("n,density", [(64, 0.8), (90, 0.7), (128, 0.55), (129, 0.5), (230, 0.35), (256, 0.3)])
def test_counts_on_both_sides_of_the_depth_line(n, density):
    G = _dense(n, density, n)
    rp, col = G.csr()
    orp, oc = O.orient(rp.astype(np.uint64), col)
    o = G.orient("degree")
    exp = {k: O.count(orp, oc, k, "pivot_tails", "node")["count"] for k in (3, 4, 5, 6, 7, 8)}
    for k, e in exp.items():
        for gran in ("node", "edge"):
            assert o.count(k, "pivot", gran, part_size=1).count == e, (k, gran)
    for ks in ((4, 5), (4, 8), (5, 6, 7)):
        for gran in ("node", "edge"):
            res, _ = K.batch_count([(o, dict(k=k, algo="pivot", gran=gran)) for k in ks])
            assert [r.count for r in res] == [exp[k] for k in ks], (ks, gran)


def _hub_task(n, density, planted, seed):
    """oriented CSR (rowptr, col, key) of a hub with arcs to the n vertices of a random graph with a planted
    near-clique: the hub's task has n vertices, the others' are small"""
    r = np.random.default_rng(seed)
    a, b = np.triu_indices(n, 1)
    keep = r.random(a.size) < density
    dense = np.zeros(n, bool)
    dense[r.choice(n, planted, replace=False)] = True
    keep |= dense[a] & dense[b] & (r.random(a.size) < 0.9)
    src = np.concatenate([np.zeros(n, np.int64), a[keep] + 1])
    dst = np.concatenate([np.arange(1, n + 1), b[keep] + 1])
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=n + 1))])
    return rowptr.astype(np.uint32), dst.astype(np.uint32), np.minimum(np.arange(n + 1), 1).astype(np.uint32)


# a task of the class above 256 vertices, above 512 and above 1024
@pytest.mark.parametrize("n,density", [(300, 0.3), (600, 0.15), (1100, 0.08)])
def test_block_wide_tasks_on_both_sides_of_the_depth_line(n, density, tmp_path):
    rowptr, col, key = _hub_task(n, density, 45, n)
    write_oriented(tmp_path / "hub.kco", rowptr, col, key, n)
    o = K.Oriented.load(str(tmp_path / "hub.kco"))
    exp = {k: O.count(rowptr.astype(np.uint64), col, k, "pivot_tails", "node")["count"] for k in (5, 6, 7, 8, 9)}
    for k, e in exp.items():
        r = o.count(k, "pivot", "node", part_size=1)
        print(n, k, r.count, round(r.raw["count_ms"], 1), flush=True)
        assert r.count == e and e > 0, k
        assert o.count_noalloc(k, "pivot", "node").count == e, k
    for k in (5, 6, 7):  # both sides in one launch
        res, _ = K.batch_count([(o, dict(k=x, algo="pivot", gran="node")) for x in (k, k + 2)])
        assert [r.count for r in res] == [exp[k], exp[k + 2]], k
