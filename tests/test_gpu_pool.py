"""GPU: which device memory the library keeps and which it gives back."""
import ctypes
import time

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
