"""A new search on the same open lists starts from the source alone: entries that the last search left
beyond its goal's cost do not pile up (they overflowed the lists after some dozens of searches)."""
import pytest

pytestmark = pytest.mark.gpu

INF = float("inf")


@pytest.mark.parametrize("kind,kw", [("lhq", dict(capacity_per_lp=64)), ("lsq", dict(capacity_per_lp=64)),
                                     ("laq", dict(capacity_per_lp=64)),
                                     ("laq", dict(capacity_per_lp=64, update_ids=97 * 61)),
                                     ("laq", dict(capacity_per_lp=32, far_per_lp=64))])
def test_searches_on_one_queue_start_empty(gpq, kind, kw):
    with gpq.Queue(kind, num_lps=64, stage_per_lp=16, lookahead=INF, horizon=INF, **kw) as q:
        a = gpq.Astar(q, 97, 61, connectivity=8, seed=3, threshold=0.2)
        costs = set()
        for _ in range(40):
            a.model_init()
            assert q.queue_check_phold() == 1
            costs.add(a.run("graph", 16)["cost"])
        assert len(costs) == 1 and q.error_flags() == 0
        a.model_finish()
