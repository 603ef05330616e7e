"""Tile searches whose tiles are entered again and again, with inboxes and parked entries of many more
records than a wave takes: every wave of a tile's workgroup has to see the inbox's length before it is
cleared for the step after next, or the cells of the others are lost without a flag and the cost
comes out too high.  Several searches on one handle; the cost is the oracle's and the path has it."""
import pytest

from test_astar_gpu import check_path, oracle_grid, thr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [16, 32])
@pytest.mark.parametrize("conn,density", [(4, 0.35), (8, 0.1), (8, 0.4)])
@pytest.mark.parametrize("window", [1, 40, 0xFFFFFFFF])
def test_inboxes_of_several_waves(gpq, oracle, tile, conn, density, window):
    w, h = 517, 389
    q = gpq.Queue("lhq", num_lps=8, capacity_per_lp=64, stage_per_lp=16, lookahead=float("inf"), horizon=float("inf"))
    for seed in (1, 2, 3, 4):
        s, t = (seed, 2), (w - 1 - seed, h - 3)
        a = gpq.Astar(q, w, h, connectivity=conn, source=s, target=t, seed=seed, threshold=density, tile=tile,
                      window=window)
        grid = oracle_grid(oracle, w, h, seed, 0, 0, thr(density), forced=(s, t))
        cost = oracle.dijkstra(grid, w, h, conn, s, t)
        for _ in range(2):
            a.model_init()
            rep = a.run(mode="graph", batch=16)
            assert rep["cost"] == cost and rep["error_flags"] == 0, (seed, tile, conn, window)
        if cost >= 0:
            check_path(a.path(), grid, w, conn, s, t, cost)
        a.model_finish()
    q.queue_finish()
