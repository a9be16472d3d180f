"""Walker counts that are no multiple of 16 move their lattices byte by byte:
team tiles of such batches take little longer than those of aligned ones (1.46
times with one byte in flight at a time, 1.02 with four; 1.25 allows for the
launch's spread), and give the lane tiles' chains."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


def test_ragged_walkers_cost_little():
    t = {}
    for W in (1784, 1792):
        with M.Batch([dict(L=32, walkers=W, seed=i, beta=1.8) for i in range(8)]) as b:
            assert b.tiles == M.KERNEL_TEAM
            b.init(0)
            t[W] = min(b.iterate_profiled(1)[0] for _ in range(6))
    assert t[1784] < 1.25 * t[1792], t


@pytest.mark.parametrize("L,W", [(8, 17), (10, 31), (32, 1000), (34, 33), (72, 5)])
def test_ragged_tiles_match_lane_tiles(L, W):
    got = []
    for tiles in (M.KERNEL_TEAM if L % 8 == 0 else M.KERNEL_AUTO, M.KERNEL_LANE):
        with M.Batch([dict(L=L, walkers=W, seed=3, init_nup=5), dict(L=L, walkers=W + 2, seed=4)],
                     tiles=tiles) as b:
            b.init(0)
            b.iterate(5)
            got.append([x for i in range(2) for x in
                        (b.get_hist(i), b.get_log_weight(i), b.get_lattice(i), *b.get_state(i))])
    for x, y in zip(*got):
        assert np.array_equal(x, y)
