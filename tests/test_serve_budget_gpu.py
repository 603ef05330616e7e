"""The serving budget against memory kept from destroyed handles: the PHOLD pool takes no kept block that is
larger than what it asks for, so the bytes it reports are the bytes it holds.  A queue of 1.8 times the
pool's LPs is destroyed first; its blocks stay kept, and the pool's own come on top."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

BUDGET = 1 << 30
SMALL = dict(seed=5, phold_fraction=0.6, phold_log2=(10, 12), phold_init_per_lp=4, phold_end_time=2.0)


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so.7")                  # the one the library has loaded
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_pool_takes_its_own_blocks(gpq):
    gpq.release_kept_memory()
    rep, first = gpq.serve_run(6, mode="graph", hbm_budget=BUDGET, **SMALL)
    assert 0 < rep["pool_bytes"] <= BUDGET
    gpq.release_kept_memory()
    lps = int(1.8 * rep["pool_bytes"] / (16 * (64 + 32 + 128)))    # ring, staging and far records of an LP
    gpq.Queue("laq", num_lps=lps, capacity_per_lp=64, stage_per_lp=32, far_per_lp=128).queue_finish()
    before = _free_bytes()
    again, second = gpq.serve_run(6, mode="graph", hbm_budget=BUDGET, **SMALL)
    assert before - _free_bytes() > 0.9 * again["pool_bytes"]
    assert again["pool_bytes"] == rep["pool_bytes"]
    assert [r["result"] for r in first] == [r["result"] for r in second]
    gpq.release_kept_memory()
