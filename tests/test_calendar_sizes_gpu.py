"""Calendars beyond the sizes that the logs with one writer take (their filing launch keeps the counts
of a group's logs in LDS): more than 2^23 LPs with 256 windows.  They use the logs with atomics.
Per-LP counts and hashes against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_more_lps_than_the_filing_launch_takes(gpq, oracle):
    lps, end = (1 << 23) + 3, 0.25
    q = gpq.Queue("laq", num_lps=lps, lookahead=0.1, horizon=end, capacity_per_lp=1, stage_per_lp=1, far_per_lp=1,
                  calendar_windows=256)
    m = gpq.Phold(q, init_per_lp=1, seed=3, drain="fused", checks=False)
    m.model_init()
    rep = gpq.des_run(m, mode="graph", batch=4)
    cnt, hsh = m.lp_state()
    pending = q.queue_check_phold()
    gpq.des_finish(m)
    gpq.release_kept_memory()
    res, ocnt, ohsh = oracle.phold("seq", lps, 1, end, seed=3)
    assert rep["events"] == res.events and pending == lps
    assert np.array_equal(cnt, ocnt) and np.array_equal(hsh, ohsh)
