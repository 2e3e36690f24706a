"""GPU: a clique whose tree walk carries more than 4,096 pivots into its last subtrees, against binomials."""
from math import comb

import numpy as np
import pytest

import kcgpu_amd as K

pytestmark = pytest.mark.gpu


def test_one_task_of_a_clique_of_4400():
    """vertex 0 of a complete graph, the largest node task, alone (a sample of the tasks)"""
    n = 4400
    a, b = np.triu_indices(n, 1)
    o = K.Graph.from_edges(a.astype(np.uint32), b.astype(np.uint32), n).orient("degree")
    assert o.info()["m"] == a.size and o.info()["max_out_degree"] == n - 1
    for k in (3, 5, 6):  # (k = 6: five vertices below the root, the tree is walked to the end of its chain)
        r = o.count_sampled(k, n, 0, "pivot", "node")
        print(k, r.count, r.raw["count_ms"], flush=True)
        assert r.count == comb(n - 1, k - 1) and r.raw["tasks"] == 1, k
