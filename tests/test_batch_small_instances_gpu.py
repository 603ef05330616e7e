"""Calendar batches of many small instances: an instance takes whole blocks of 256 LPs, not of 512, when
units of 512 would mostly hold LPs that nobody uses; on both sides of the rule.  Hashes and counts
against the oracle, and the memory of the batch against its blocks'."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _check(oracle, inst, hashes, events, every):
    for i, (lps, k, seed, end) in enumerate(inst):
        if i % every == 0 or i == len(inst) - 1:
            res, _, _ = oracle.phold("seq", lps, k, end, seed=seed)
            assert events[i] == res.events and hashes[i] == res.trace_hash, i


@pytest.mark.parametrize("sizes", [
    [250] * 900,                    # 256 LPs each, 512 in units: blocks
    [600] * 400,                    # a third more in units, few LPs: blocks
    [2100] * 100,                   # a ninth more: units
    [700] * 700,                    # a third more, from 2^19 LPs on: units
    [1, 511, 512, 513, 255, 256, 257] * 120,
])
def test_instances_in_blocks_or_units(gpq, oracle, sizes):
    inst = [(lps, 3, 1000 + i, 1.0 + (i % 3) * 0.5) for i, lps in enumerate(sizes)]
    with gpq.PholdBatch(inst, calendar_windows=64, capacity_per_lp=8, stage_per_lp=4, far_per_lp=8) as b:
        b.run("graph", batch=8)
        hashes, events = b.results()
    _check(oracle, inst, hashes, events, 37)


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so.7")                  # the one the library has loaded
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_memory_of_small_instances(gpq, oracle):
    n, windows, cap, far, stage = 3000, 64, 8, 32, 4
    inst = [(10, 3, i + 1, 1.0) for i in range(n)]
    gpq.release_kept_memory()
    before = _free_bytes()
    with gpq.PholdBatch(inst, calendar_windows=windows, capacity_per_lp=cap, stage_per_lp=stage, far_per_lp=far) as b:
        b.run("graph", batch=8)
        hashes, events = b.results()
    held = before - _free_bytes()          # kept for the next batch
    gpq.release_kept_memory()
    # per LP: logs, three lists, staging, a two-record ring, 64 bytes of words; the log counters
    per_lp = 16 * (windows * cap + 3 * far + stage + 2) + 64 + windows * 64 // 256
    assert held < 1.25 * n * 256 * per_lp, (held, n * 256 * per_lp)
    _check(oracle, inst, hashes, events, 500)
