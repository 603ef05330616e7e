"""Ties of the batched A*: on an open 4-connected grid every cell between the endpoints has the goal's f.
Entries taken newest first reach the goal in about as many iterations as the path has steps, of at
most a workgroup's cells each; taken oldest first they fill the whole rectangle before."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("side,threads", [(1024, 64), (2048, 128)])
def test_open_grid_expands_a_band(gpq, side, threads):
    S = gpq._lib.QuerySpec
    specs = [S(side, 0, 0, 0, side - 1, side - 1, 4, 1, 1, 0), S(side, 0, side - 1, 0, 0, side - 1, 4, 1, 1, 1)]
    steps = 2 * (side - 1)
    with gpq.AstarBatch(specs, threads_per_query=threads) as b:
        b.run("graph")
        costs, expanded = b.results()
    assert list(costs) == [steps, steps]
    # an even band is threads * steps; twice that is a quarter of the cells
    assert 4 * threads * steps <= side * side
    assert max(expanded) <= 2 * threads * steps, expanded
