"""The record sort at the edges of its levels (one run of 1024, 128 runs, 128 x 128 runs) and on inputs
that strain the 128-way merges: every key equal, few distinct keys, sorted, reversed, runs that
interleave, and records that equal the padding word for word.  Records are compared whole; equal
keys are ordered by dst."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sort(gpq, a):
    out = np.zeros_like(a)
    p = gpq._ptr
    gpq._lib.check(gpq.lib.gpq_selftest_sort(p(a), len(a), p(out)), "sort")
    return out


def _make(gpq, n, how):
    rng = np.random.default_rng(n)
    a = np.zeros(n, dtype=gpq.event_dtype)
    a["dst"] = rng.permutation(n).astype(np.uint32)
    if how == "equal":
        a["ts"], a["src"], a["seq"] = 7, 3, 5
    elif how == "few":
        a["ts"], a["src"], a["seq"] = rng.integers(0, 2, n), rng.integers(0, 2, n), rng.integers(0, 3, n)
    elif how == "sorted":
        a["ts"] = np.arange(n)
    elif how == "reversed":
        a["ts"] = np.arange(n)[::-1]
    elif how == "interleaved":
        a["ts"] = np.arange(n) % 1024
        a["src"] = np.arange(n) // 1024
    elif how == "ones":
        a["ts"], a["src"], a["seq"] = 0xFFFFFFFF, 0xFFFFFFFF, 0xFFFFFFFF
        a["dst"][::2] = 0xFFFFFFFF
    else:
        a["ts"] = rng.exponential(1.0, n).astype(np.float32).view(np.uint32)
        a["src"], a["seq"] = rng.integers(0, 50, n), rng.integers(0, 1 << 32, n, dtype=np.uint64)
    return a


@pytest.mark.parametrize("how", ["equal", "few", "sorted", "reversed", "interleaved", "ones", "random"])
@pytest.mark.parametrize("n", [1, 33, 1023, 1024, 1025, 4097, 131071, 131072, 131073, 262177])
def test_sort_at_level_edges(gpq, n, how):
    a = _make(gpq, n, how)
    want = a[np.lexsort((a["dst"], a["seq"], a["src"], a["ts"]))]
    assert np.array_equal(_sort(gpq, a), want)


def test_sort_three_levels(gpq):
    n = (1 << 24) + 33
    a = _make(gpq, n, "random")
    out = _sort(gpq, a)
    key = lambda e: (e["ts"].astype(np.uint64) << np.uint64(32)) | e["src"]
    k = key(out)
    assert np.all(k[:-1] <= k[1:])
    same = k[:-1] == k[1:]
    assert np.all(out["seq"][:-1][same] <= out["seq"][1:][same])
    assert np.array_equal(np.sort(out["dst"]), np.arange(n))              # every record once, whole:
    back = np.zeros_like(a)
    back[out["dst"]] = out
    src = np.zeros_like(a)
    src[a["dst"]] = a
    assert np.array_equal(back, src)


@pytest.mark.parametrize("how", ["equal", "interleaved", "random"])
@pytest.mark.parametrize("n", [163841, 393217, 524288, 700001, 1048575, 1048576, 1048577, 4194304, 4194305])
def test_sort_of_two_narrow_levels(gpq, n, how):
    # up to 2^20 records the two levels merge up to 32 runs each, up to 2^22 64, above it 128
    a = _make(gpq, n, how)
    want = a[np.lexsort((a["dst"], a["seq"], a["src"], a["ts"]))]
    assert np.array_equal(_sort(gpq, a), want)
