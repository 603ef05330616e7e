"""The global queues' selection and merge when a launch's blocks take more than one tile each: a
scanned prefix of more than 1024 tiles of 1024 records, a merge of more than 1024 tiles, and prefixes
that end at a tile's edge.  Every run commits the oracle's trace."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,L,k,la,T,kw", [
    ("gaq", 1300003, 2, 4.0, 1.5, dict(total_capacity=3 * 1300003, stage_per_lp=1)),
    ("hq", 1300003, 2, 4.0, 1.0, dict(capacity_per_lp=6, stage_per_lp=1, node_size=1300003)),
    ("gaq", 1023, 1, 4.0, 3.0, dict(capacity_per_lp=8, stage_per_lp=2)),     # one tile less a record, ...
    ("gaq", 1024, 1, 4.0, 3.0, dict(capacity_per_lp=8, stage_per_lp=2)),
    ("gaq", 1025, 1, 4.0, 3.0, dict(capacity_per_lp=8, stage_per_lp=2)),
    ("gaq", 1, 1, 4.0, 3.0, dict(capacity_per_lp=8, stage_per_lp=2)),
])
def test_long_prefix_keeps_the_trace(gpq, oracle, kind, L, k, la, T, kw):
    q = gpq.Queue(kind, num_lps=L, lookahead=la, horizon=T, **kw)
    m = gpq.Phold(q, init_per_lp=k, seed=42, end_time=T)
    m.model_init()
    rep = gpq.des_run(m, mode="graph", batch=8)
    res, cnt, hsh = oracle.phold("seq", L, k, T, lookahead=la)
    c, h = m.lp_state()
    assert q.error_flags() == 0
    assert rep["events"] == res.events and m.trace_hash() == res.trace_hash
    assert np.array_equal(c, cnt) and np.array_equal(h, hsh)
    m.model_finish()
    q.queue_finish()
