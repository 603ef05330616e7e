"""Kept memory after many handles: a thousand queues alive at once leave some ten thousand kept blocks, and
making the next queue does not search them all."""
import time

import pytest

pytestmark = pytest.mark.gpu


def _make(gpq):
    return gpq.Queue("lhq", num_lps=64, capacity_per_lp=16, stage_per_lp=8, lookahead=0.1, horizon=5.0)


def _median_create(gpq, rounds=41):
    times = []
    for _ in range(rounds):
        t = time.perf_counter()
        _make(gpq).queue_finish()
        times.append(time.perf_counter() - t)
    return sorted(times)[rounds // 2]


def test_creating_a_queue_after_a_thousand(gpq):
    gpq.release_kept_memory()
    few = _median_create(gpq)
    queues = [_make(gpq) for _ in range(1500)]
    for q in queues:
        q.queue_finish()
    many = _median_create(gpq)
    gpq.release_kept_memory()
    assert many < 4 * few + 100e-6, (few, many)
