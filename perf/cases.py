"""The work that users of this package have it do, as timed cases.

A case is a dict of plain values.  Its "path" names the public route it takes:

  phold        one whole PHOLD simulation: des_init, model_init, des_run (hipGraph replays), the per-LP
               counts and trace hashes read back, des_finish.  "layout" picks the event list.  A model
               cannot be run twice, so a program that sweeps seeds makes this whole sequence each time.
  phold_batch  many simulations of uneven size in one calendar (PholdBatch), results read back
  astar        one grid query on a kept Astar handle: model_init (grid, source), run, optimal cost
  astar_batch  independent grid queries in one persistent launch on a kept AstarBatch, optimal costs
  serve        a saturated trace of mixed simulations and queries through serve_run
  sort         the allocation-free record sort, device records to device records

Every output is a whole number, fixed by the inputs: committed-event counts, trace hashes, path costs
and sorted records.  The order in which a search expands cells is not an output.
"""
import heapq
import math

import numpy as np
import torch

import gpupq_amd as gpq

INF = float("inf")


# ---- the event lists ------------------------------------------------------------------------
# Queue arguments per layout, and the Phold drain argument.
def _queue_args(layout, lps):
    if layout == "calendar":            # the default of bench.py
        return dict(kind="laq", capacity_per_lp=8, stage_per_lp=32, far_per_lp=128, calendar_windows=64), "fused"
    if layout == "ring_fused":          # two-tier sorted rings, merge and commit in one kernel
        return dict(kind="laq", capacity_per_lp=64, stage_per_lp=32, far_per_lp=128), "fused"
    if layout == "ring":                # two-tier sorted rings, queue_post kernel and drain step
        return dict(kind="laq", capacity_per_lp=64, stage_per_lp=32, far_per_lp=128), True
    if layout == "lhq":                 # binary heaps, each LP's safe window per step
        return dict(kind="lhq", capacity_per_lp=128, stage_per_lp=32), True
    if layout == "lsq":                 # splay trees, each LP's safe window per step
        return dict(kind="lsq", capacity_per_lp=128, stage_per_lp=32), True
    if layout == "gaq":                 # one global sorted array, one event per LP and step
        return dict(kind="gaq", capacity_per_lp=64, stage_per_lp=2), False
    if layout == "hq":                  # one parallel heap, a node holds an event per LP
        return dict(kind="hq", capacity_per_lp=40, stage_per_lp=1, node_size=max(lps, 32)), False
    raise ValueError("layout %r" % layout)


def listed():
    return [
        # the smallest useful simulation (bench.py's phold_1024_k16_t100): a thousand dependent
        # windows of about 1500 events each, where the latency of a step is all there is
        dict(name="phold_1k", path="phold", layout="calendar", lps=1024, k=16, end=100.0, lookahead=0.1, p_self=0.5),
        # the benchmark's own simulation: 2^25 events in flight, 1.5e9 committed
        dict(name="phold_1m", path="phold", layout="calendar", lps=1 << 20, k=32, end=50.0, lookahead=0.1,
             p_self=0.5),
        # the general local array queue (any model can be written on its verbs), an uneven LP count
        dict(name="phold_ring", path="phold", layout="ring", lps=200003, k=16, end=20.0, lookahead=0.1, p_self=0.5),
        # the splay queue, an uneven LP count
        dict(name="phold_lsq", path="phold", layout="lsq", lps=100003, k=16, end=20.0, lookahead=0.1, p_self=0.5),
        # the global sorted array: a large array, few new events per step
        dict(name="phold_gaq", path="phold", layout="gaq", lps=250007, k=32, end=5.0, lookahead=0.1, p_self=0.5),
        # the parallel heap, a medium model
        dict(name="phold_hq", path="phold", layout="hq", lps=100003, k=16, end=10.0, lookahead=0.1, p_self=0.5),
        # a sweep: 32 simulations of 2^12 to 2^18 LPs advanced together (bench.py's phold_batch)
        dict(name="phold_batch", path="phold_batch", instances=32, lo=12.0, hi=18.0, k=16, end=20.0, lookahead=0.1),
        # one query on the benchmark's 4096 x 4096 grid, searched by tiles
        dict(name="astar_tiles", path="astar", lists=64, queue="lhq", tile=32, width=4096, height=4096,
             connectivity=4, density=0.2),
        # one query on open lists in heaps, 8-connected, an odd grid
        dict(name="astar_lists", path="astar", lists=4096, queue="lhq", tile=0, width=1001, height=703,
             connectivity=8, density=0.2),
        # 512 queries of uneven size (sides 256 to 2048) in one launch (bench.py's astar_batch)
        dict(name="astar_batch", path="astar_batch", queries=512, threads=512, stage=8),
        # 64 mixed requests arriving at once: serving under full load
        dict(name="serve", path="serve", requests=64, phold_fraction=0.5, lo=12, hi=18, k=16, end=20.0),
        # the record sort inside a caller's own step, an odd number of records
        dict(name="sort", path="sort", records=100003),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges; costs no more than phold_1m."""
    path = rng.choice(["phold", "phold", "phold", "phold_batch", "astar", "astar", "astar_batch", "serve", "sort"])
    if path == "phold":
        layout = rng.choice(["calendar", "calendar", "ring_fused", "ring", "lhq", "lsq", "gaq", "hq"])
        # the largest LP counts by how fast an event list is
        top = {"calendar": 1 << 20, "ring_fused": 400000, "ring": 400000, "lhq": 200000, "lsq": 100000,
               "gaq": 250000, "hq": 100000}[layout]
        lps = _log_uniform(rng, 700, top)
        k = rng.choice([4, 8, 16, 24, 32])
        lookahead = rng.choice([0.05, 0.1, 0.2]) if k <= 16 else 0.1
        end = {"gaq": 5.0, "hq": 5.0, "lsq": 10.0}.get(layout, 20.0) * rng.uniform(0.5, 1.0)
        return dict(path="phold", layout=layout, lps=lps, k=k, end=round(end, 2), lookahead=lookahead,
                    p_self=rng.choice([0.2, 0.5, 0.8]))
    if path == "phold_batch":
        return dict(path="phold_batch", instances=rng.randint(2, 40), lo=round(rng.uniform(9.0, 12.0), 2),
                    hi=round(rng.uniform(14.0, 17.5), 2), k=rng.choice([8, 16]), end=round(rng.uniform(8.0, 20.0), 2),
                    lookahead=0.1)
    if path == "astar":
        con = rng.choice([4, 8])
        tile = rng.choice([0, 16, 32])
        top = 1024 if tile == 0 else 3000
        w, h = _log_uniform(rng, 100, top), _log_uniform(rng, 100, top)
        return dict(path="astar", lists=rng.choice([4096, 16384]), queue=rng.choice(["lhq", "laq"]), tile=tile,
                    width=w, height=h, connectivity=con, density=round(rng.uniform(0.1, 0.3), 3))
    if path == "astar_batch":
        return dict(path="astar_batch", queries=_log_uniform(rng, 20, 512), threads=rng.choice([256, 512]), stage=8)
    if path == "serve":
        return dict(path="serve", requests=rng.randint(8, 64), phold_fraction=round(rng.uniform(0.3, 0.7), 2), lo=11,
                    hi=rng.choice([16, 17, 18]), k=rng.choice([8, 16]), end=round(rng.uniform(8.0, 20.0), 2))
    return dict(path="sort", records=_log_uniform(rng, 600, 1 << 20))


# ---- inputs -----------------------------------------------------------------------------------
def _rng(seed):
    return np.random.default_rng(np.random.SeedSequence([20, seed & 0xFFFFFFFF]))


def _seed31(rng):
    return int(rng.integers(1, 2 ** 31 - 1))


def _instances(case, rng):
    return [(int(round(2 ** rng.uniform(case["lo"], case["hi"]))), case["k"], _seed31(rng), case["end"],
             case["lookahead"]) for _ in range(case["instances"])]


def _query(case, rng):
    """Obstacle seed, and endpoints near opposite corners (within a sixteenth of each side)."""
    w, h = case["width"], case["height"]
    seed31 = _seed31(rng)
    sx, tx = int(rng.integers(0, w // 16 + 1)), w - 1 - int(rng.integers(0, w // 16 + 1))
    sy, ty = int(rng.integers(0, h // 16 + 1)), h - 1 - int(rng.integers(0, h // 16 + 1))
    return seed31, (sx, sy), (tx, ty)


def _records(case, rng):
    """Events as a PHOLD step schedules them: Exp(1) + lookahead timestamps, (src, seq) unique."""
    n = case["records"]
    ev = np.zeros(n, dtype=gpq.event_dtype)
    ev["ts"] = (rng.exponential(1.0, n).astype(np.float32) + np.float32(0.1)).view(np.uint32)
    ev["dst"] = rng.integers(0, max(n, 1), n, dtype=np.uint32)
    ev["src"] = rng.permutation(n).astype(np.uint32)
    ev["seq"] = rng.integers(0, 1000, n, dtype=np.uint32)
    return ev


def prepare(case, seed):
    rng = _rng(seed)
    st = {"case": case}
    path = case["path"]
    if path == "phold":
        st["seed"] = _seed31(rng)
    elif path == "phold_batch":
        st["batch"] = gpq.PholdBatch(_instances(case, rng), calendar_windows=64, capacity_per_lp=8, stage_per_lp=32,
                                     far_per_lp=32)
    elif path == "astar":
        if case["queue"] == "lhq":      # a binary heap per open list
            kw = dict(capacity_per_lp=256)
        else:                           # short sorted rings backed by far stores
            kw = dict(capacity_per_lp=64, far_per_lp=512)
        q = gpq.Queue(case["queue"], num_lps=case["lists"], stage_per_lp=32, lookahead=INF, horizon=INF, **kw)
        st["queue"] = q
        seed31, source, target = _query(case, rng)
        st["astar"] = gpq.Astar(q, case["width"], case["height"], connectivity=case["connectivity"], source=source,
                                target=target, seed=seed31, threshold=case["density"], tile=case["tile"])
    elif path == "astar_batch":
        master = _seed31(rng)
        specs = [gpq.query_synthetic(master, i) for i in range(case["queries"])]
        st["batch"] = gpq.AstarBatch(specs, threads_per_query=case["threads"], stage_capacity=case["stage"])
    elif path == "serve":
        st["args"] = dict(seed=_seed31(rng), rate=0.0, phold_fraction=case["phold_fraction"], hbm_budget=8 << 30,
                          phold_log2=(case["lo"], case["hi"]), phold_init_per_lp=case["k"],
                          phold_end_time=case["end"])
    else:
        ev = _records(case, rng)
        st["in"] = torch.from_numpy(ev.view(np.int32).reshape(-1, 4).copy()).cuda()
        st["out"] = torch.empty_like(st["in"])
    return st


# ---- one pass ---------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    path = case["path"]
    if path == "phold":
        args, drain = _queue_args(case["layout"], case["lps"])
        q = gpq.des_init(num_lps=case["lps"], lookahead=case["lookahead"], horizon=case["end"], **args)
        m = gpq.Phold(q, init_per_lp=case["k"], seed=state["seed"], p_self=case["p_self"], checks=False, drain=drain)
        m.model_init()
        rep = gpq.des_run(m, mode="graph", batch=64)
        counts, hashes = m.lp_state()
        gpq.des_finish(m)
        return {"events": rep["events"], "counts": counts, "hashes": hashes}
    if path == "phold_batch":
        state["batch"].run("graph", batch=16)
        hashes, events = state["batch"].results()
        return {"hashes": hashes, "events": events}
    if path == "astar":
        a = state["astar"]
        a.model_init()
        return {"cost": a.run("graph", 32)["cost"]}
    if path == "astar_batch":
        state["batch"].run("graph")
        return {"costs": state["batch"].results()[0]}
    if path == "serve":
        _, reqs = gpq.serve_run(case["requests"], mode="graph", **state["args"])
        return {"result": np.array([r["result"] for r in reqs], dtype=np.uint64),
                "events": np.array([r["work"] if r["kind"] == 0 else 0 for r in reqs], dtype=np.uint64)}
    status = gpq.lib.gpq_sort_events_noalloc(state["in"].data_ptr(), case["records"], state["out"].data_ptr(),
                                             torch.cuda.current_stream().cuda_stream)
    if status != 0:
        raise RuntimeError("gpq_sort_events_noalloc: status %d" % status)
    return {"sorted": state["out"]}


# ---- work -------------------------------------------------------------------------------------
EVENT_BYTES = 32       # a 16-byte record is written once when scheduled and read once when due
EVENT_OPS = 130        # ten Philox rounds, the exponential, the trace hash


def _events(lps, k, end, lookahead):
    """Expected committed events: each of the lps * k events in flight recurs every 1 + lookahead."""
    return lps * k * (end + lookahead) / (1.0 + lookahead)


def work(case):
    path = case["path"]
    if path == "phold":
        e = _events(case["lps"], case["k"], case["end"], case["lookahead"])
        return {"bytes": EVENT_BYTES * e + 12.0 * case["lps"], "flops": EVENT_OPS * e}
    if path == "phold_batch":
        span = (case["hi"] - case["lo"]) * math.log(2.0)
        lps = case["instances"] * (2 ** case["hi"] - 2 ** case["lo"]) / span
        e = _events(lps, case["k"], case["end"], case["lookahead"])
        return {"bytes": EVENT_BYTES * e + 12.0 * lps, "flops": EVENT_OPS * e}
    if path == "astar":
        # a query across a uniformly cluttered grid closes about half of the cells: the obstacle
        # bit of each cell, and a path cost written per closed cell
        cells = case["width"] * case["height"]
        return {"bytes": cells / 8.0 + 4.0 * cells / 2.0, "flops": 4.0 * case["connectivity"] * cells / 2.0}
    if path == "astar_batch":
        cells = case["queries"] * (2048.0 ** 2 - 256.0 ** 2) / (2.0 * math.log(8.0))
        return {"bytes": cells / 8.0 + 4.0 * cells / 4.0, "flops": 32.0 * cells / 4.0}
    if path == "serve":
        np_ = case["requests"] * case["phold_fraction"]
        na = case["requests"] - np_
        lps = np_ * (2.0 ** case["hi"] - 2.0 ** case["lo"]) / ((case["hi"] - case["lo"]) * math.log(2.0))
        e = _events(lps, case["k"], case["end"], 0.1)
        cells = na * (2048.0 ** 2 - 256.0 ** 2) / (2.0 * math.log(8.0))
        return {"bytes": EVENT_BYTES * e + 12.0 * lps + cells * (1 / 8.0 + 1.0), "flops": EVENT_OPS * e + 8.0 * cells}
    n = case["records"]
    return {"bytes": 32.0 * n, "flops": n * max(math.log2(n), 1.0)}


# ---- the values, computed independently ---------------------------------------------------------
def _philox(c0, c1, c2, c3, key):
    """Philox4x32-10 (Salmon et al., SC'11) of counters (c0 array, c1, c2, c3) under key (key, 0)."""
    m0, m1, lo32 = np.uint64(0xD2511F53), np.uint64(0xCD9E8D57), np.uint64(0xFFFFFFFF)
    x = [np.broadcast_to(np.asarray(c, dtype=np.uint64), c0.shape).copy() for c in (c0, c1, c2, c3)]
    k0, k1 = key & 0xFFFFFFFF, 0
    for _ in range(10):
        p0, p1 = m0 * x[0], m1 * x[2]
        x = [(p1 >> np.uint64(32)) ^ x[1] ^ np.uint64(k0), p1 & lo32,
             (p0 >> np.uint64(32)) ^ x[3] ^ np.uint64(k1), p0 & lo32]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return x


def _obstacles(width, height, seed, density, source, target):
    """Obstacle map with a border of obstacles (height + 2, width + 2); the endpoints are free."""
    n = width * height
    words = _philox(np.arange((n + 3) // 4, dtype=np.uint64), 0, 0, 2, seed)
    blocked = (np.stack(words, axis=1).reshape(-1)[:n] < np.uint64(min(int(density * 2 ** 32), 0xFFFFFFFF)))
    for x, y in (source, target):
        blocked[y * width + x] = False
    g = np.ones((height + 2, width + 2), dtype=bool)
    g[1:-1, 1:-1] = blocked.reshape(height, width)
    return g


def _cost(case, seed31, source, target):
    """Optimal path cost by Dial's algorithm, one numpy step per cost and neighbour."""
    w, h = case["width"], case["height"]
    closed = _obstacles(w, h, seed31, case["density"], source, target).reshape(-1)
    s = w + 2
    src, dst = ((y + 1) * s + x + 1 for x, y in (source, target))
    if case["connectivity"] == 4:
        moves = [(1, 1), (-1, 1), (s, 1), (-s, 1)]
    else:
        moves = [(1, 10), (-1, 10), (s, 10), (-s, 10), (s + 1, 14), (s - 1, 14), (-s + 1, 14), (-s - 1, 14)]
    buckets, costs = {0: [np.array([src])]}, [0]
    while costs:
        c = heapq.heappop(costs)
        f = np.unique(np.concatenate(buckets.pop(c)))
        f = f[~closed[f]]
        if not f.size:
            continue
        closed[f] = True
        if closed[dst]:
            return c
        for d, step in moves:
            nb = f + d
            nb = nb[~closed[nb]]
            if nb.size:
                if c + step not in buckets:
                    buckets[c + step] = []
                    heapq.heappush(costs, c + step)
                buckets[c + step].append(nb)
    return -1


def exact(case, seed):
    """Sorted records and single-query costs.  Counts and hashes of a simulation are defined by its
    float32 timestamps, and have no value of more digits; batches of queries take too long here."""
    if case["path"] == "sort":
        ev = _records(case, _rng(seed))
        ev = ev[np.lexsort((ev["seq"], ev["src"], ev["ts"]))]
        return {"sorted": torch.from_numpy(ev.view(np.int32).reshape(-1, 4).copy())}
    if case["path"] == "astar":
        return {"cost": _cost(case, *_query(case, _rng(seed)))}
    return None
