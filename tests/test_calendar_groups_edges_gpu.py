"""The filing launch of large calendars past the sizes it takes at once: more than 2048 units, whose
outboxes are looked at in turns, and more than 8192 events for one group in a step.  Per-LP counts and
hashes against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lps,k,end,lookahead,windows,cap,far,p_self", [
    ((1 << 20) + 1, 1, 0.5, 0.1, 8, 2, 2, 0.0),          # 2049 units: the last one alone in its turn
    ((1 << 21) + 700, 1, 0.4, 0.1, 16, 2, 2, 0.5),       # two whole turns and two units
    (196608 + 300, 32, 3.0, 1.0, 8, 64, 64, 0.0),        # some 16 events per LP and step, all for other LPs
])
def test_turns_of_the_filing_launch(gpq, oracle, lps, k, end, lookahead, windows, cap, far, p_self):
    q = gpq.Queue("laq", num_lps=lps, lookahead=lookahead, horizon=end, capacity_per_lp=cap, stage_per_lp=4,
                  far_per_lp=far, calendar_windows=windows)
    m = gpq.Phold(q, init_per_lp=k, seed=8, p_self=p_self, drain="fused")
    m.model_init()
    rep = gpq.des_run(m, mode="graph", batch=4)
    cnt, hsh = m.lp_state()
    pending = q.queue_check_phold()
    gpq.des_finish(m)
    res, ocnt, ohsh = oracle.phold("seq", lps, k, end, seed=8, lookahead=lookahead,
                                   p_self_u32=min(int(round(p_self * 2 ** 32)), 0xFFFFFFFF))
    assert rep["events"] == res.events and pending == lps * k
    assert np.array_equal(cnt, ocnt) and np.array_equal(hsh, ohsh)
