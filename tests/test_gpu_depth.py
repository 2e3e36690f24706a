"""GPU: pivoting at the line between the register kernels without and with matrix operands (five vertices below a
task's root: k = 7 for edge tasks, 6 for node tasks), alone and with both sides of it in one launch."""
import numpy as np
import pytest

import kcgpu_amd as K
from oracle import oracle as O

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
