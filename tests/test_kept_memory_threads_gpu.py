"""Kept memory shared by host threads: every round of every thread completes and gives the oracle's
trace.  An exception in a thread, a thread that does not end or a round that is missing fails the
test."""
import threading
import traceback

import numpy as np
import pytest

from test_kept_memory_gpu import LAYOUTS, _simulate

pytestmark = pytest.mark.gpu

THREADS, ROUNDS = 6, 3


def test_every_round_of_every_thread(gpq, oracle):
    _, cnt, hsh = oracle.phold("seq", 1500, 8, 6.0, seed=9)
    done, failed = [], []

    def work(i):
        try:
            for r in range(ROUNDS):
                c, h = _simulate(gpq, LAYOUTS[(i + r) % len(LAYOUTS)])
                if np.array_equal(c, cnt) and np.array_equal(h, hsh):
                    done.append((i, r))
                else:
                    failed.append("thread %d round %d: another trace" % (i, r))
                if r == 1 and i % 2:
                    gpq.release_kept_memory()              # while the others allocate
        except BaseException:
            failed.append("thread %d: %s" % (i, traceback.format_exc()))

    threads = [threading.Thread(target=work, args=(i,), daemon=True) for i in range(THREADS)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=100)
    assert not failed, "\n".join(failed)
    assert not any(t.is_alive() for t in threads)
    assert sorted(done) == [(i, r) for i in range(THREADS) for r in range(ROUNDS)]
