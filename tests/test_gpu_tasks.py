"""GPU: how tasks are dealt to waves and binned, at the sizes where it can go wrong."""
import numpy as np
import pytest

import kcgpu_amd as K

pytestmark = pytest.mark.gpu


def _disjoint_cliques(sizes):
    """edge list of disjoint cliques of the given sizes, and the vertex count"""
    src, dst, at = [], [], 0
    for s, times in sizes:
        a, b = np.triu_indices(s, 1)
        base = at + s * np.arange(times, dtype=np.int64)[:, None]
        src.append((base + a).ravel())
        dst.append((base + b).ravel())
        at += s * times
    return np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32), at


# around the queue count (32), the one-task-per-block grid and four tasks per grab
@pytest.mark.parametrize("t", [1, 31, 32, 33, 64, 2047, 8191, 8192, 8193, 100_003, 524_288, 524_289, 600_001])
def test_every_task_is_taken_once(t):
    src, dst, n = _disjoint_cliques([(4, t)])
    o = K.orient_edges(src, dst, "degree", n=n)
    for algo in ("pivot", "orient"):
        r = o.count(4, algo, "node", part_size=1)  # one task of three vertices per clique
        assert r.count == t and r.raw["tasks"] == t, algo
    r = o.count(4, "pivot", "edge", part_size=1)
    assert r.count == t and r.raw["tasks"] == t
