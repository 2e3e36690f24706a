"""GPU: calls that are refused after work was queued, and the calls that follow on the same device blocks."""
import struct

import numpy as np
import pytest

import kcgpu_amd as K
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def write_oriented(path, rowptr, col, key, max_out):
    """an oriented-CSR cache file (format of Oriented.save)"""
    h = 14695981039346656037
    for b in b"".join(np.ascontiguousarray(x, dtype="<u4").tobytes() for x in (rowptr, col, key)):
        h = ((h ^ b) * 1099511628211) & (2 ** 64 - 1)
    with open(path, "wb") as f:
        f.write(struct.pack("<8sIIQIIQ", b"KCOCSR1\0", key.size, 0, col.size, max_out, 0, h))
        for x in (rowptr, col, key):
            f.write(np.ascontiguousarray(x, dtype="<u4").tobytes())


def test_refused_count_leaves_nothing_running(tmp_path):
    """a task of 70,000 vertices is more than the block-wide kernel takes: the count is refused once the tasks are
    binned, and orientations and counts right after it are right"""
    leaves = 70_000
    rowptr = np.full(leaves + 2, leaves, np.uint32)
    rowptr[0] = 0
    key = np.ones(leaves + 1, np.uint32)
    key[0] = 0
    write_oriented(tmp_path / "star.kco", rowptr, np.arange(1, leaves + 1, dtype=np.uint32), key, leaves)
    G = K.Graph.generate(K.GEN_CHUNG_LU, seed=5, n=20_000, m=130_000, gamma=2.1, max_degree=900)
    rp, col = G.csr()
    orp, oc = O.orient(rp.astype(np.uint64), col, O.peel_priority(rp.astype(np.uint64), col)[0])
    exp = O.count(orp, oc, 5, "pivot_tails", "node")["count"]
    for _ in range(3):
        star = K.Oriented.load(str(tmp_path / "star.kco"))
        for _ in range(2):
            with pytest.raises(K.KCError) as e:
                star.count(4, "pivot", "node")
            assert e.value.code == K.KC_ERR_LIMIT
        assert star.count(3, "pivot", "edge").count == 0
        star.close()
        o = G.orient("degen")
        assert o.count(5, "pivot", "node").count == exp
        with pytest.raises(K.KCError):
            K.orient_edges(np.array([0, 9], np.uint32), np.array([1, 2], np.uint32), "degree", n=5)  # an id beyond n
        assert o.count(5, "pivot", "edge").count == exp
        o.close()
