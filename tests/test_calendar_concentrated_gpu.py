"""Large calendars whose initial events concentrate on a few LPs: the events beyond the calendar may lie
anywhere as long as they fit the queue as a whole (num_lps * far_per_lp of them), although every group
of LPs has a list of its own.  Extra initial events come through the host's queue_insert; the trace
is that of a plain event loop over the oracle's random numbers and hash."""
import heapq

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LPS, FAR, SEED, LOOKAHEAD = 196608 + 5, 4, 6, np.float32(0.1)
HALF = 0x80000000


def _event_loop(oracle, end, extra):
    """(counts, hashes) of PHOLD with one initial event per LP and `extra` ones."""
    exp = oracle.exp_table()
    bits = lambda f: int(np.float32(f).view(np.uint32))
    end_bits = bits(end)
    heap = [(int(t), int(s), int(q), int(d)) for t, d, s, q in extra.tolist() if t < end_bits]
    for lp in range(LPS):
        t = bits(exp[oracle.philox((0, lp, 1, 0), (SEED, 0))[0] >> 8])
        if t < end_bits:
            heap.append((t, lp, 0, lp))
    heapq.heapify(heap)
    cnt, hsh = np.zeros(LPS, dtype=np.uint32), np.zeros(LPS, dtype=np.uint64)
    while heap:
        t, src, seq, lp = heapq.heappop(heap)
        n = int(cnt[lp])
        hsh[lp] = oracle.trace_step(int(hsh[lp]), t, src, seq)
        cnt[lp] += 1
        r = oracle.philox((n, lp, 0, 0), (SEED, 0))
        now = np.uint32(t).view(np.float32)
        t2 = bits(np.float32(now + LOOKAHEAD) + exp[r[0] >> 8])
        if t2 < end_bits:
            heapq.heappush(heap, (t2, lp, 1 + n, lp if r[1] < HALF else (r[2] * LPS) >> 32))
    return cnt, hsh


def _extra(gpq, first, lps, per_lp, lo, hi):
    rng = np.random.default_rng(2)
    ev = np.zeros(lps * per_lp, dtype=gpq.event_dtype)
    ev["ts"] = rng.uniform(lo, hi, len(ev)).astype(np.float32).view(np.uint32)
    ev["dst"] = ev["src"] = np.repeat(np.arange(first, first + lps), per_lp)
    ev["seq"] = 1000000 + np.arange(len(ev))
    return ev


def _queue(gpq, windows, end, far=FAR):
    return gpq.Queue("laq", num_lps=LPS, lookahead=float(LOOKAHEAD), horizon=end, capacity_per_lp=8, stage_per_lp=16,
                     far_per_lp=far, calendar_windows=windows)


@pytest.mark.parametrize("windows,end,lps,lo,hi", [
    (8, 1.5, 1024, 0.0, 8.0),        # two groups, most events beyond the calendar and the end
    (16, 1.75, 1024, 1.0, 4.0),
    (8, 1.0, 700, 0.0, 2.0),
])
def test_concentrated_initial_events(gpq, oracle, windows, end, lps, lo, hi):
    first, per_lp = 5000, 32
    ev = _extra(gpq, first, lps, per_lp, lo, hi)
    with _queue(gpq, windows, end) as q:
        half = np.arange(len(ev)) % per_lp < per_lp // 2          # a staging row at a time
        for part in (ev[half], ev[~half]):
            q.insert(part)
            q.queue_post_init()
        assert q.error_flags() == 0 and q.queue_check_phold() == len(ev)
        assert len(q.lp_contents(first + lps - 1)) == per_lp
        m = gpq.Phold(q, init_per_lp=1, seed=SEED, drain="fused")
        m.model_init()
        assert q.error_flags() == 0 and q.queue_check_phold() == LPS + len(ev)
        assert len(q.lp_contents(first + lps - 1)) == per_lp + 1
        rep = gpq.des_run(m, mode="graph", batch=4)
        cnt, hsh = m.lp_state()
        assert q.queue_check_phold() == LPS + len(ev)
        m.model_finish()
    ocnt, ohsh = _event_loop(oracle, end, ev)
    assert rep["events"] == int(ocnt.sum()) and rep["error_flags"] == 0
    assert np.array_equal(cnt, ocnt) and np.array_equal(hsh, ohsh)


def test_more_events_than_the_queue_holds_are_flagged(gpq):
    ev = _extra(gpq, 0, 20000, 16, 0.5, 4.0)
    with _queue(gpq, 8, 1.0, far=1) as q:
        m = gpq.Phold(q, init_per_lp=1, seed=SEED, drain="fused")
        q.insert(ev)
        q.queue_post_init()
        with pytest.raises(gpq.GpqError, match="capacity"):
            m.model_init()
        assert q.error_flags() & 2
        m.model_finish()
