"""Local splay queues across repeated deletes of the minimum: chains, equal keys, one-node trees and trees
that empty and fill again, against a sorted model."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["up", "down", "mixed", "equal"])
@pytest.mark.parametrize("count", [1, 2, 3, 17, 64])
def test_minima_in_order(gpq, order, count):
    lps = 65
    rng = np.random.default_rng(count)
    with gpq.Queue("lsq", num_lps=lps, capacity_per_lp=64, stage_per_lp=64, lookahead=1e9, horizon=float("inf")) as q:
        for rnd in range(2):                            # the second round fills emptied trees
            want = {}
            a = np.zeros(count * lps, dtype=gpq.event_dtype)
            for lp in range(lps):
                ts = {"up": np.arange(count), "down": np.arange(count)[::-1], "mixed": rng.integers(0, 8, count),
                      "equal": np.zeros(count, dtype=int)}[order]
                for i in range(count):
                    # equal keys differ in nothing; mixed ones in source and number
                    src, seq = (0, 0) if order == "equal" else (int(rng.integers(0, 3)), i)
                    a[lp * count + i] = (gpq.f32_bits(float(ts[i])), lp, src, seq)
                    want.setdefault(lp, []).append((gpq.f32_bits(float(ts[i])), src, seq))
            q.insert(a)
            q.queue_post()
            got = {lp: [] for lp in range(lps)}
            for step in range(count):
                items, _ = q.peek(set_done=True)
                assert len(items) == lps
                for e in items:
                    got[int(e["dst"])].append((int(e["ts"]), int(e["src"]), int(e["seq"])))
                if step % 5 == 0:
                    q.queue_post()                      # nothing staged: the trees stay
            for lp in range(lps):
                assert got[lp] == sorted(want[lp]), (rnd, lp)
            assert q.queue_check_phold() == 0 and q.error_flags() == 0
