"""GPU: which device memory the library keeps and which it gives back."""
import ctypes
import time
from math import comb

import numpy as np
import pytest

import kcgpu_amd as K

pytestmark = pytest.mark.gpu


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_removed_graphs_leave_the_device():
    """a server's graph, and what its orientation took, leave the device with kc_server_remove_graph"""
    small = K.Graph.generate(K.GEN_BA, seed=1, n=3000, attach=8)
    big = K.Graph.generate(K.GEN_ER, seed=2, n=400_000, m=8_000_000)
    srv = K.Server(workers=1)
    try:
        for mode in ("degree", "degen"):
            for _ in range(2):  # (code objects, streams)
                g = srv.add_graph(small, mode)
                assert srv.wait(srv.submit(g, 4)).count > 0
                srv.remove_graph(g)
            before = _free_bytes()
            g = srv.add_graph(big, mode)
            assert before - _free_bytes() >= 64 << 20
            srv.remove_graph(g)
            t0 = time.perf_counter()  # (the driver reports freed memory a little later)
            while before - _free_bytes() > 16 << 20 and time.perf_counter() - t0 < 10.0:
                time.sleep(0.05)
            print(mode, before, _free_bytes(), f"{time.perf_counter() - t0:.2f} s", flush=True)
            assert before - _free_bytes() <= 16 << 20
    finally:
        srv.close()


def test_graphs_of_the_calls_beside_a_server_are_pooled():
    """the pool serves kc_orient and kc_count next to a running server, with the same counts"""
    G = K.Graph.generate(K.GEN_BA, seed=3, n=20_000, attach=9)
    exp = G.orient("degen").count(5, "pivot", "node").count
    srv = K.Server(workers=2)
    try:
        g = srv.add_graph(G, "degen")
        for _ in range(10):
            t = [srv.submit(g, 5, algo, "node") for algo in ("pivot", "orient")]
            o = G.orient("degen")
            assert o.count(5, "pivot", "edge").count == exp
            o.close()
            assert all(srv.wait(x).count == exp for x in t)
    finally:
        srv.close()


def _pairs_graph(parts):
    """all edges between `parts` pairs of vertices but none inside a pair"""
    a, b = np.triu_indices(2 * parts, 1)
    keep = a // 2 != b // 2
    return K.Graph.from_edges(a[keep].astype(np.uint32), b[keep].astype(np.uint32), 2 * parts)


def test_adjacency_words_never_make_a_call_fail(monkeypatch):
    """on a full device (KC_DEVICE_LIMIT_MIB) a count that fits without adjacency words fits with them allowed, its own
    or another handle's, and every count that succeeds is right"""
    parts, k = 530, 4
    G = _pairs_graph(parts)  # 18 MB of words, 200 MB of slices for its tasks above 512 vertices
    other = K.Graph.generate(K.GEN_CHUNG_LU, seed=8, n=300_000, m=1_900_000, gamma=2.1, max_degree=6000)

    def fits(limit, words):
        monkeypatch.setenv("KC_WORDS_MIB", words)
        monkeypatch.setenv("KC_DEVICE_LIMIT_MIB", str(limit))
        o = None
        try:
            o = G.orient("degree")
            for _ in range(2):
                assert o.count(k, "pivot", "node").count == comb(parts, k) << k
            return True
        except K.KCError as e:
            assert e.code == K.KC_ERR_NOMEM
            return False
        finally:
            if o:
                o.close()

    least = next(x for x in range(0, 4096, 32) if fits(x, "0"))
    for limit in range(max(0, least - 32), least + 40, 2):  # on both sides of what it needs
        without = fits(limit, "0")
        assert fits(limit, "2048") or not without, limit

    monkeypatch.delenv("KC_DEVICE_LIMIT_MIB")
    monkeypatch.setenv("KC_WORDS_MIB", "0")
    o = other.orient("degen")
    exp = o.count(6, "pivot", "edge").count
    least = next(x for x in range(0, 4096, 4) if fits(x, "0"))
    for _ in range(2):  # now it holds 60 MB of words, until the other graph's count wants them
        monkeypatch.delenv("KC_DEVICE_LIMIT_MIB")
        monkeypatch.setenv("KC_WORDS_MIB", "2048")
        assert o.count(6, "pivot", "edge").count == exp
        assert fits(least, "0")
    monkeypatch.setenv("KC_DEVICE_LIMIT_MIB", str(least))
    assert o.count(6, "pivot", "edge").count == exp and o.count(6, "pivot", "node").count == exp


def test_edge_list_that_leaves_no_room_for_the_ranks(monkeypatch):
    """the CSR build with and without the places of the edge ends: from the least memory it takes upwards"""
    r = np.random.default_rng(3)
    ne, n = 1_000_003, 60_000
    s, d = (np.minimum(r.zipf(1.4, ne), n) - 1).astype(np.uint32), r.integers(0, n, ne, dtype=np.uint32)
    exp = K.Graph.from_edges(s, d, n).csr()

    def fits(limit):
        monkeypatch.setenv("KC_DEVICE_LIMIT_MIB", str(limit))
        try:
            rp, col = K.Graph.from_edges_device(s, d, n).csr()
        except K.KCError as e:
            assert e.code == K.KC_ERR_NOMEM
            return False
        assert (rp == exp[0]).all() and (col == exp[1]).all()
        return True

    least = next(x for x in range(0, 4096, 1) if fits(x))
    for limit in range(least, least + 14):  # (8 MB of ranks)
        assert fits(limit), limit
