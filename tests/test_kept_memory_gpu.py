"""Memory kept from destroyed handles: a simulation gives the oracle's trace whatever the blocks it
takes held before (another queue kind's records, a grid search's costs), before and after the kept
blocks are freed, and from several host threads at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

INF = float("inf")
LAYOUTS = [
    ("laq", dict(capacity_per_lp=8, stage_per_lp=32, far_per_lp=32, calendar_windows=64), "fused"),
    ("laq", dict(capacity_per_lp=64, stage_per_lp=32, far_per_lp=128), True),
    ("lhq", dict(capacity_per_lp=128, stage_per_lp=32), True),
    ("lsq", dict(capacity_per_lp=128, stage_per_lp=32), True),
    ("gaq", dict(capacity_per_lp=64, stage_per_lp=2), False),
    ("hq", dict(capacity_per_lp=40, stage_per_lp=1, node_size=1500), False),
]


def _simulate(gpq, layout, lps=1500):
    kind, kw, drain = layout
    q = gpq.Queue(kind, num_lps=lps, lookahead=0.1, horizon=6.0, **kw)
    m = gpq.Phold(q, init_per_lp=8, seed=9, drain=drain)
    m.model_init()
    gpq.des_run(m, mode="graph", batch=16)
    st = m.lp_state()
    gpq.des_finish(m)
    return st


def test_blocks_change_hands(gpq, oracle):
    _, cnt, hsh = oracle.phold("seq", 1500, 8, 6.0, seed=9)
    for turn in range(2):
        for layout in LAYOUTS:
            c, h = _simulate(gpq, layout)
            assert np.array_equal(c, cnt) and np.array_equal(h, hsh), (turn, layout)
            with gpq.Queue("lhq", num_lps=256, capacity_per_lp=64, stage_per_lp=16, lookahead=INF, horizon=INF) as q:
                costs = set()
                for tile in (0, 16):
                    a = gpq.Astar(q, 90, 70, connectivity=8, seed=5, threshold=0.2, tile=tile)
                    a.model_init()
                    costs.add(a.run("graph", 8)["cost"])
                    a.model_finish()
                assert len(costs) == 1
        gpq.release_kept_memory()


def test_threads_share_the_kept_blocks(gpq, oracle):
    _, cnt, hsh = oracle.phold("seq", 1500, 8, 6.0, seed=9)
    bad = []

    def work(i):
        for r in range(3):
            c, h = _simulate(gpq, LAYOUTS[(i + r) % len(LAYOUTS)])
            if not (np.array_equal(c, cnt) and np.array_equal(h, hsh)):
                bad.append((i, r))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(timeout=100)
    assert not bad
