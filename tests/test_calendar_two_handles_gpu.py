"""Two large calendars at once: the filing launch of the first needs more LDS for its counts than that of
the second, which is created after it (64 and 32 KiB).  Per-LP counts and hashes against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_a_smaller_calendar_leaves_the_larger_its_lds(gpq, oracle):
    sizes, end, pairs = ((1 << 22) + 1, (1 << 21) + 1), 0.5, []
    for lps in sizes:
        q = gpq.Queue("laq", num_lps=lps, lookahead=0.1, horizon=end, capacity_per_lp=1, stage_per_lp=1, far_per_lp=1,
                      calendar_windows=256)
        pairs.append((q, gpq.Phold(q, init_per_lp=1, seed=4, drain="fused", checks=False)))
    for (_, m), lps in zip(pairs, sizes):
        m.model_init()
        rep = gpq.des_run(m, mode="graph", batch=4)
        cnt, hsh = m.lp_state()
        res, ocnt, ohsh = oracle.phold("seq", lps, 1, end, seed=4)
        assert rep["events"] == res.events
        assert np.array_equal(cnt, ocnt) and np.array_equal(hsh, ohsh)
    for _, m in pairs:
        gpq.des_finish(m)
    gpq.release_kept_memory()
