"""Two-tier rings whose runs are shorter and longer than the two register slots of the narrow merge pass,
in one wave and in different ones: PHOLD with few and many events per LP commits the oracle's trace."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [32, 128])
@pytest.mark.parametrize("k,p_self", [(1, 0.5), (7, 0.0), (16, 0.5), (40, 1.0), (60, 0.5)])
@pytest.mark.parametrize("lps", [63, 257])
def test_ring_lengths(gpq, oracle, cap, k, p_self, lps):
    if cap == 32 and k > 16:
        pytest.skip("more events than a 32-slot ring takes")
    T = 6.0
    q = gpq.Queue("laq", num_lps=lps, capacity_per_lp=cap, stage_per_lp=64, far_per_lp=512, lookahead=0.1, horizon=T)
    m = gpq.Phold(q, init_per_lp=k, seed=5, end_time=T, p_self=p_self)
    m.model_init()
    rep = gpq.des_run(m, mode="graph", batch=16)
    res, cnt, hsh = oracle.phold("seq", lps, k, T, seed=5, p_self_u32=min(int(p_self * 2 ** 32), 0xFFFFFFFF))
    c, h = m.lp_state()
    assert q.error_flags() == 0
    assert rep["events"] == res.events and m.trace_hash() == res.trace_hash
    assert np.array_equal(c, cnt) and np.array_equal(h, hsh)
    m.model_finish()
    q.queue_finish()
