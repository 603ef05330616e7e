"""The parallel heap's merge launches: node sizes around a merge tile, as many insert chunks as a
step may have, several heaps, and nodes so large that some merges of a step take a partition launch
and others do not.  Every run commits the oracle's trace and leaves a heap."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,r,k,T,heaps,tile", [
    (5, 1, 6, 4.0, 1, 1024),              # a record per node, chunks for every insert
    (700, 100, 8, 6.0, 1, 0),             # eight chunks, deep heap
    (700, 100, 8, 6.0, 3, 0),
    (2047, 2047, 8, 4.0, 1, 0), (2048, 2048, 8, 4.0, 1, 0), (2049, 2049, 8, 4.0, 2, 0),
    (3001, 1023, 12, 4.0, 1, 1024), (3001, 1025, 12, 4.0, 1, 4096),
    (360001, 360001, 2, 0.6, 1, 0),       # 3 r reaches the partition launch, 2 r does not
])
def test_heap_trace_and_order(gpq, oracle, L, r, k, T, heaps, tile):
    if L * 1 > 7 * r:
        pytest.skip("more inserts than chunks")
    nodes = -(-(-(-L // heaps) * max(40, 2 * k)) // r) + 9
    q = gpq.Queue("hq", num_lps=L, node_size=r, heap_nodes=nodes, stage_per_lp=1, lookahead=0.1, horizon=T, heaps=heaps,
                  sort_tile=tile)
    m = gpq.Phold(q, init_per_lp=k, seed=42, end_time=T)
    m.model_init()
    rep = gpq.des_run(m, mode="graph", batch=16)
    res, cnt, hsh = oracle.phold("seq", L, k, T)
    c, h = m.lp_state()
    assert q.error_flags() == 0
    assert rep["events"] == res.events and m.trace_hash() == res.trace_hash
    assert np.array_equal(c, cnt) and np.array_equal(h, hsh)

    def key(e):
        return (int(e["ts"]), int(e["src"]), int(e["seq"]))
    held = 0
    for hp in range(heaps):
        ends = []
        for v in range(nodes):
            a = q.heap_node(hp * nodes + v)
            held += len(a)
            if len(a) > 1:
                rec = a.astype(a.dtype)
                order = np.lexsort((rec["seq"], rec["src"], rec["ts"]))
                assert np.array_equal(order, np.arange(len(a))), "node %d is not sorted" % v
            ends.append((key(a[0]), key(a[-1])) if len(a) else None)
            if v and ends[v] and ends[(v - 1) // 2]:
                assert ends[(v - 1) // 2][1] <= ends[v][0], "node %d before its parent" % v
    assert held == q.queue_check_phold()
    m.model_finish()
    q.queue_finish()
