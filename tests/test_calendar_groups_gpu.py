"""Large calendars (logs with one writer, a filing launch before each commit): the smallest size that
takes that path, sizes that end inside a unit and a group, passes over long logs, few windows
(most events wait beyond the calendar), and instances sharing one calendar.  Per-LP counts and
hashes against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIN = 196608


def _sim(gpq, lps, k, end, lookahead, windows, cap, far, p_self):
    q = gpq.Queue("laq", num_lps=lps, lookahead=lookahead, horizon=end, capacity_per_lp=cap, stage_per_lp=4,
                  far_per_lp=far, calendar_windows=windows)
    m = gpq.Phold(q, init_per_lp=k, seed=3, p_self=p_self, drain="fused")
    m.model_init()
    return q, m


@pytest.mark.parametrize("lps,k,end,lookahead,windows,cap,far,p_self", [
    (MIN, 4, 3.0, 0.1, 64, 8, 16, 0.5),
    (MIN + 1, 2, 3.0, 0.1, 8, 8, 4, 0.5),            # one LP in the last unit; most events beyond 8 windows
    (MIN + 513, 20, 3.0, 0.5, 16, 64, 32, 0.5),      # seven events per LP and window: two passes over a log
    (300001, 3, 2.0, 0.1, 256, 8, 16, 0.0),          # every event for another LP
    (MIN + 700, 3, 2.0, 0.1, 64, 8, 16, 1.0),        # every event for its own LP: empty outboxes
    (MIN - 1, 4, 2.0, 0.1, 64, 8, 16, 0.5),          # the largest calendar with atomics
])
def test_large_calendar_matches_oracle(gpq, oracle, lps, k, end, lookahead, windows, cap, far, p_self):
    q, m = _sim(gpq, lps, k, end, lookahead, windows, cap, far, p_self)
    rep = gpq.des_run(m, mode="graph", batch=8)
    cnt, hsh = m.lp_state()
    pending = q.queue_check_phold()
    gpq.des_finish(m)
    res, ocnt, ohsh = oracle.phold("seq", lps, k, end, seed=3, lookahead=lookahead,
                                   p_self_u32=min(int(round(p_self * 2 ** 32)), 0xFFFFFFFF))
    assert rep["events"] == res.events and pending == lps * k
    assert np.array_equal(cnt, ocnt) and np.array_equal(hsh, ohsh)


def test_contents_between_steps(gpq, oracle):
    lps, k = MIN + 5, 3
    q, m = _sim(gpq, lps, k, 2.0, 0.1, 8, 8, 16, 0.5)
    for _ in range(4):
        m.model_handle_next()
        q.queue_post()
        assert q.queue_check_phold() == lps * k
        for lp in (0, 4711, lps - 1):
            c = q.lp_contents(lp)
            key = [(int(e["ts"]), int(e["src"]), int(e["seq"])) for e in c]
            assert key == sorted(key) and all(int(e["dst"]) == lp for e in c) and q.queue_length(lp) == len(c)
    rep = gpq.des_run(m, mode="plain")
    res, _, _ = oracle.phold("seq", lps, k, 2.0, seed=3)
    assert rep["events"] == res.events and m.trace_hash() == res.trace_hash
    gpq.des_finish(m)


def test_instances_share_a_large_calendar(gpq, oracle):
    inst = [(150000, 6, 5, 3.0), (100, 5, 6, 2.0), (50001, 4, 7, 1.0), (1, 3, 8, 3.0)]
    with gpq.PholdBatch(inst, calendar_windows=64, capacity_per_lp=8, stage_per_lp=4, far_per_lp=16) as b:
        b.run("graph", batch=8)
        hashes, events = b.results()
    for i, (lps, k, seed, end) in enumerate(inst):
        res, _, _ = oracle.phold("seq", lps, k, end, seed=seed)
        assert events[i] == res.events and hashes[i] == res.trace_hash
