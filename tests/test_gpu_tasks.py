"""GPU: how tasks are dealt to waves and binned, at the sizes where it can go wrong."""
from math import comb

import numpy as np
import pytest
import scipy.sparse as sp

import kcgpu_amd as K
from oracle import oracle as O

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


def _oracle_count(G, mode, k, gran):
    rp, col = G.csr()
    rp = rp.astype(np.uint64)
    orp, oc = O.orient(rp, col, O.peel_priority(rp, col)[0] if mode == "degen" else None)
    return O.count(orp, oc, k, "pivot_tails", gran)["count"]


# candidate sets at the edges of the 32- and 64-vertex words, of the matrix blocks and of the register classes
@pytest.mark.parametrize("n", [5, 6, 31, 32, 33, 34, 63, 64, 65, 66, 96, 97, 128, 129, 130, 160, 200])
@pytest.mark.parametrize("density", [0.3, 0.7, 0.93])
def test_dense_random_graphs_vs_oracle(n, density):
    r = np.random.default_rng(n * 100 + int(density * 100))
    a, b = np.triu_indices(n, 1)
    keep = r.random(a.size) < density
    G = K.Graph.from_edges(a[keep].astype(np.uint32), b[keep].astype(np.uint32), n)
    o = G.orient("degree")
    for k in (4, 5) + ((6,) if n <= 130 else ()) + ((7, 8) if n <= 66 else ()):
        exp = _oracle_count(G, "degree", k, "node")
        for gran in ("node", "edge"):
            r = o.count(k, "pivot", gran, part_size=1)
            assert r.count == exp, (k, gran)


# 11 node tasks above 128 vertices a clique: on both sides of the line between one wave and one block a task
@pytest.mark.parametrize("cliques", [1, 325, 326])
def test_tasks_above_128_vertices_few_and_many(cliques):
    src, dst, n = _disjoint_cliques([(140, cliques)])
    o = K.orient_edges(src, dst, "degree", n=n)
    for k in (4, 6, 9):
        assert o.count(k, "pivot", "node", part_size=1).count == cliques * comb(140, k)


# out-lists much longer than the tasks (pair by pair) and about as long (entry by entry)
@pytest.mark.parametrize("n,m,hub", [(3000, 40_000, 900), (20_000, 120_000, 4000), (20_000, 40_000, 50)])
@pytest.mark.parametrize("mode", ["degree", "degen"])
def test_bitmaps_of_short_tasks_in_long_rows(n, m, hub, mode):
    G = K.Graph.generate(K.GEN_CHUNG_LU, seed=n + m, n=n, m=m, gamma=2.1, max_degree=hub)
    o = G.orient(mode)
    for k, gran in ((4, "node"), (4, "edge"), (5, "edge")):
        exp = _oracle_count(G, mode, k, gran)
        for algo in ("pivot", "orient"):
            assert o.count(k, algo, gran, part_size=1).count == exp, (k, gran, algo)


def test_device_blocks_are_reused():
    """graphs of several sizes oriented, counted and freed in turn, twice over the same device blocks"""
    for i in range(20):
        t = 50 + 400 * (i % 5)
        src, dst, n = _disjoint_cliques([(7, t), (3, i + 1)])
        G = K.Graph.from_edges(src, dst, n)
        for mode in ("degree", "degen"):
            o = G.orient(mode)
            assert o.count(5, "pivot", "edge", part_size=1).count == t * 21
            rp, col, key = o.export()
            assert int(rp[-1]) == col.size == 21 * t + 3 * (i + 1) and key.size == n
            o.close()


def _edge_list_graphs():
    """out-lists around the hash's sizes (512, 256), 16-lane groups and 64-edge chunks"""
    yield "cliques", [(s, 1) for s in (3, 16, 17, 18, 33, 64, 65, 66, 128, 257, 258, 512, 513, 514, 515, 600)]
    yield "chunk63", [(2, 63), (3, 1)]
    yield "chunk64", [(2, 64), (4, 1)]
    yield "many", [(3, 5001), (5, 700), (2, 31)]


@pytest.mark.parametrize("name,sizes", list(_edge_list_graphs()))
def test_triangles_over_edge_tasks(name, sizes):
    src, dst, n = _disjoint_cliques(sizes)
    o = K.orient_edges(src, dst, "degree", n=n)
    exp = sum(comb(s, 3) * t for s, t in sizes)
    tasks = sum(comb(s - 1, 2) * t for s, t in sizes)  # edges whose list has a member
    for algo in ("pivot", "orient"):
        r = o.count(3, algo, "edge", part_size=1)
        assert r.count == exp and r.raw["tasks"] == tasks
        assert sum(o.count_sampled(3, 5, f, algo, "edge").count for f in range(5)) == exp
    assert o.count_noalloc(3, "pivot", "edge").count == exp
    assert o.count(4, "pivot", "edge", part_size=1).count == sum(comb(s, 4) * t for s, t in sizes)


@pytest.mark.parametrize("mode", ["degree", "degen"])
def test_triangles_over_edge_tasks_vs_oracle(mode):
    for kind, kw in ((K.GEN_RMAT, dict(scale=12, edge_factor=12, a=0.57, b=0.19, c=0.19)),
                     (K.GEN_CHUNG_LU, dict(n=30_000, m=200_000, gamma=2.1, max_degree=3000)),
                     (K.GEN_ER, dict(n=5000, m=60_000))):
        G = K.Graph.generate(kind, seed=11, **kw)
        rp, col = G.csr()
        rp = rp.astype(np.uint64)
        orp, oc = O.orient(rp, col, O.peel_priority(rp, col)[0] if mode == "degen" else None)
        exp = O.count(orp, oc, 3, "pivot", "edge")
        r = G.orient(mode).count(3, "pivot", "edge", part_size=1)
        assert (r.count, r.raw["tasks"]) == (exp["count"], exp["tasks"])
        # bytes: the two list heads and both lists of every edge whose lists meet (no bitmap is built at k = 3)
        d = np.diff(orp.astype(np.int64))
        A = sp.csr_matrix((np.ones(oc.size, np.int64), oc, orp.astype(np.int64)), shape=(d.size, d.size))
        met = A.multiply(A @ A.T).tocoo()
        assert r.raw["alg_bytes"] == int((24 + 4 * (d[met.row] + d[met.col])).sum())


# per-vertex counts of tasks at the edges of one word, where one count goes through both kernels
@pytest.mark.parametrize("n", [4, 5, 33, 64, 65, 66, 90, 128, 129, 130, 140])
@pytest.mark.parametrize("density", [0.3, 0.8, 1.0])
def test_local_counts_at_word_edges_vs_oracle(n, density):
    r = np.random.default_rng(n)
    a, b = np.triu_indices(n, 1)
    keep = r.random(a.size) < density
    G = K.Graph.from_edges(a[keep].astype(np.uint32), b[keep].astype(np.uint32), n)
    rp, col = G.csr()
    orp, oc = O.orient(rp.astype(np.uint64), col)
    o = G.orient("degree")
    for k in (3, 4, 5, 6, 9):
        exp, ovf = O.count_local(orp, oc, k, "pivot_tails", "node")
        assert not ovf
        for gran in ("node", "edge"):
            loc, tot = o.count_local(k, "pivot", gran)
            assert (loc == exp).all() and tot.count * k == int(exp.sum(dtype=np.uint64)), (k, gran)


# tasks whose rows come from the adjacency words of the size pass, on both sides of the list lengths that
# decide it (32, 256) and of the words and half words of T; a batch of two queries takes the lists
@pytest.mark.parametrize("sizes", [(31, 32, 33, 34, 35), (64, 65, 66, 67), (96, 97, 98), (128, 129, 130, 131),
                                   (192, 193, 194, 195), (255, 256, 257, 258, 259), (400,)])
@pytest.mark.parametrize("density", [0.15, 0.9])
def test_tasks_from_adjacency_words_equal_lists(sizes, density):
    r = np.random.default_rng(sum(sizes))
    src, dst, at = [], [], 0
    for n in sizes:
        a, b = np.triu_indices(n, 1)
        keep = r.random(a.size) < density
        keep |= (a == 0) | (a == n // 2)  # two vertices with long lists either way
        p = at + r.permutation(n)
        src.append(p[a[keep]])
        dst.append(p[b[keep]])
        at += n
    s, d = np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32)
    G = K.Graph.from_edges(s, d, at)
    for mode in ("degree", "degen"):
        o = G.orient(mode)
        for k in (4, 5, 6):
            both, _ = K.batch_count([(o, dict(k=k, algo="pivot", gran="edge"))] * 2)
            one = [o.count(k, "pivot", "edge") for _ in range(2)]
            for x in one:
                assert x.count == both[0].count == both[1].count == o.count(k, "pivot", "node").count
            loc, tot = o.count_local(k, "pivot", "edge")
            ref, _ = o.count_local(k, "pivot", "node")
            assert (loc == ref).all() and tot.count == one[0].count
            for gran in ("edge", "node"):
                parts = [o.count_sampled(k, 3, i, "pivot", gran) for i in range(3)]  # (lists too)
                one = o.count(k, "pivot", gran)
                for what in ("count", "tasks", "alg_bytes"):
                    assert sum(x.raw[what] for x in parts) == one.raw[what], (k, gran, what)
                if k == 4 and sizes[-1] < 300:  # the orientation's search over the same rows
                    for P in (1, 8, 64):
                        assert o.count(k, "orient", gran, part_size=P).count == one.count
                    if sizes[-1] < 100:
                        assert (o.count_local(k, "orient", gran)[0] == ref).all()
