"""The tile search where its words and halos meet the grid's edges: widths that are not whole words or
tiles, one-cell-wide grids, and grids on both sides of the line between the two ways to find the next
window (more tiles than one block takes).  The cost is the oracle's and the path has it."""
import pytest

from test_astar_gpu import check_path, oracle_grid, thr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile", [16, 32])
@pytest.mark.parametrize("conn", [4, 8])
@pytest.mark.parametrize("w,h", [(1, 70), (70, 1), (31, 33), (32, 32), (33, 31), (63, 65), (97, 15), (257, 129)])
def test_tile_search_at_the_edges(gpq, oracle, tile, conn, w, h):
    for window in (0, 3, 0xFFFFFFFF):
        q = gpq.Queue("lhq", num_lps=8, capacity_per_lp=64, stage_per_lp=16, lookahead=float("inf"),
                      horizon=float("inf"))
        s, t = (0, 0), (w - 1, h - 1)
        a = gpq.Astar(q, w, h, connectivity=conn, source=s, target=t, seed=3, threshold=0.15, tile=tile, window=window)
        a.model_init()
        rep = a.run(mode="graph", batch=8)
        grid = oracle_grid(oracle, w, h, 3, 0, 0, thr(0.15), forced=(s, t))
        cost = oracle.dijkstra(grid, w, h, conn, s, t)
        assert rep["cost"] == cost and rep["error_flags"] == 0, (w, h, conn, tile, window)
        if cost >= 0:
            check_path(a.path(), grid, w, conn, s, t, cost)
        a.model_finish()
        q.queue_finish()


def test_tile_search_with_more_tiles_than_one_block_takes(gpq, oracle):
    w, h = 2560, 2576                                      # 160 x 161 tiles of 16: 25,760
    q = gpq.Queue("lhq", num_lps=8, capacity_per_lp=64, stage_per_lp=16, lookahead=float("inf"), horizon=float("inf"))
    a = gpq.Astar(q, w, h, connectivity=4, source=(3, 3), target=(700, 650), seed=11, threshold=0.2, tile=16)
    a.model_init()
    rep = a.run(mode="graph", batch=16)
    grid = oracle_grid(oracle, w, h, 11, 0, 0, thr(0.2), forced=((3, 3), (700, 650)))
    assert rep["cost"] == oracle.dijkstra(grid, w, h, 4, (3, 3), (700, 650)) and rep["error_flags"] == 0
    a.model_finish()
    q.queue_finish()
