"""The calendar step's commit blocks at their edges: logs longer than one pass over them (passes over
ranges of LPs), LPs with many events in one window, one LP in the last block, and equal
timestamps (a lookahead so large that float32 times coincide).  Per-LP counts and hashes against
the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lps,k,end,lookahead,cap,p_self", [
    (256, 32, 3.0, 0.1, 64, 0.5),        # several events per LP and window
    (257, 60, 2.0, 0.1, 64, 0.5),        # the last block holds one LP; 257 * 60 events
    (700, 40, 4.0, 0.5, 64, 0.5),        # 13 events per LP and window: passes over ranges of LPs
    (300, 100, 2.0, 0.25, 64, 0.9),      # 20 per LP and window, LPs with up to 64 of them
    (2, 20, 6.0, 0.1, 64, 0.5),
    (1, 4, 5.0, 0.1, 64, 1.0),
    (1025, 16, 2100.0, 100.0, 64, 0.5),  # times in the thousands: float32 steps of 1e-4, equal times
])
def test_commit_blocks_match_oracle(gpq, oracle, lps, k, end, lookahead, cap, p_self):
    q = gpq.Queue("laq", num_lps=lps, lookahead=lookahead, horizon=end, capacity_per_lp=cap, stage_per_lp=8,
                  far_per_lp=128, calendar_windows=16)
    m = gpq.Phold(q, init_per_lp=k, seed=11, p_self=p_self, drain="fused")
    m.model_init()
    rep = gpq.des_run(m, mode="graph", batch=8)
    cnt, hsh = m.lp_state()
    pending = q.queue_check_phold()
    gpq.des_finish(m)
    res, ocnt, ohsh = oracle.phold("seq", lps, k, end, seed=11, lookahead=lookahead,
                                    p_self_u32=min(int(round(p_self * 2 ** 32)), 0xFFFFFFFF))
    assert rep["events"] == res.events and pending == lps * k
    assert np.array_equal(cnt, ocnt) and np.array_equal(hsh, ohsh)
