"""GPU: how tasks are dealt to waves and binned, at the sizes where it can go wrong."""
from math import comb

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


# tasks of every size class and at the class edges, task counts around a binning tile (512 or 4,096 tasks)
@pytest.mark.parametrize("fill", [0, 500, 4096, 4097, 70_001, 600_000])
@pytest.mark.parametrize("algo", ["pivot", "orient"])
def test_binning_of_all_classes(algo, fill):
    sizes = [(s, 1) for s in (3, 17, 64, 65, 66, 128, 129, 130, 257, 258, 300, 513, 514)] + [(2, fill)]
    src, dst, n = _disjoint_cliques([x for x in sizes if x[1]])
    o = K.orient_edges(src, dst, "degree", n=n)
    for k in (3, 4):
        exp = sum(comb(s, k) * t for s, t in sizes)
        ran = {"node": sum(sum(d >= k - 1 for d in range(s)) * t for s, t in sizes),
               "edge": sum(comb(s - k + 2, 2) * t for s, t in sizes if s >= k)}
        for gran in ("node", "edge"):
            r = o.count(k, algo, gran, part_size=8)
            assert r.count == exp, (k, gran)
            assert r.raw["tasks"] == ran[gran], (k, gran)


def test_binning_of_many_queries():
    """queries of both algorithms and granularities whose tasks share binning tiles"""
    parts = [[(4, 1)], [(70, 2)], [(5, 1000), (2, 3000)], [(130, 1), (3, 1400)], [(2, 1)], [(300, 1)]]
    os_, exp = [], []
    for sizes in parts:
        src, dst, n = _disjoint_cliques(sizes)
        os_.append(K.orient_edges(src, dst, "degree", n=n))
    pairs = []
    for i in range(48):
        j, k = i % len(parts), 3 + i % 3
        pairs.append((os_[j], dict(k=k, algo=("pivot", "orient")[i % 2], gran=("node", "edge")[i // 2 % 2], part_size=1)))
        exp.append(sum(comb(s, k) * t for s, t in parts[j]))
    res, _ = K.batch_count(pairs)
    assert [r.count for r in res] == exp
