"""The batched A*'s bucketed open list where it can go wrong: buckets that fill up and spill into the
far store (a small heap_capacity on an open grid, where whole regions share one f), f ranges wider
than the row of buckets (long detours), and workgroups of the smallest and largest size.  Costs are
whole numbers and equal the oracle's Dijkstra."""
import pytest

pytestmark = pytest.mark.gpu


def _grid(oracle, s):
    g = oracle.grid(s.side, s.side, s.seed, s.stream_tag, s.query, s.threshold).copy()
    g[s.sy * s.side + s.sx] = 0
    g[s.ty * s.side + s.tx] = 0
    return g


@pytest.mark.parametrize("mode", ["graph", "plain"])
@pytest.mark.parametrize("threads,heap_capacity,stage", [(64, 256, 8), (64, 2048, 64), (256, 64, 8), (1024, 64, 4)])
def test_costs_through_spills_and_scans(gpq, oracle, threads, heap_capacity, stage, mode):
    S = gpq._lib.QuerySpec

    def thr(p):
        return int(p * 2 ** 32)

    specs = [
        S(400, 0, 30, 200, 399, 210, 8, 1, 1, 0),            # open: a wide band of cells shares each f
        S(400, 0, 30, 200, 399, 210, 4, 1, 1, 1),
        S(160, thr(0.39), 0, 0, 159, 159, 4, 5, 1, 2),       # near the percolation threshold: long detours
        S(160, thr(0.58), 0, 0, 159, 159, 8, 6, 1, 3),
        S(97, thr(0.3), 96, 0, 0, 96, 8, 7, 1, 4),
        S(33, thr(0.9), 1, 1, 30, 30, 8, 8, 1, 5),           # unreachable: the list runs empty
        S(2, 0, 0, 0, 1, 1, 4, 8, 1, 6),
    ]
    if mode == "plain":
        specs = specs[2:]
    with gpq.AstarBatch(specs, threads_per_query=threads, heap_capacity=heap_capacity, stage_capacity=stage) as b:
        b.run(mode)
        costs, _ = b.results()
    for q, s in enumerate(specs):
        want = oracle.dijkstra(_grid(oracle, s), s.side, s.side, s.connectivity, (s.sx, s.sy), (s.tx, s.ty))
        assert costs[q] == want, "query %d" % q
