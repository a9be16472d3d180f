"""E, D and M of given lattices (the state kernel) against plain numpy sums,
at the edges of its strips of 8 columns, its 32 parts per workgroup and its
groups of 32 or 128 walkers."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [2, 3, 7, 8, 9, 16, 33, 72, 250, 257])
@pytest.mark.parametrize("W", [1, 4, 31, 33, 128, 132, 254])
def test_state_matches_numpy(L, W):
    if L > 100 and W > 33:
        pytest.skip("covered by the smaller walker counts")
    rng = np.random.default_rng(1000 * L + W)
    # an ordered walker (largest byte counts), a full one, and random ones
    s = rng.integers(-1, 2, (L, L, W)).astype(np.int8)
    s[:, :, 0] = -1
    if W > 3:
        s[:, :, 2] = 1
        s[:, :, 3] = 1 - 2 * ((np.arange(L)[:, None] + np.arange(L)) % 2)
    with M.Context(L, W) as ctx:
        ctx.set_lattice(s.reshape(L * L, W))
        ctx.compute_state()
        E, D, Mg = ctx.get_state()
    a = s.astype(np.int64)
    assert np.array_equal(E, -(a * (np.roll(a, -1, 0) + np.roll(a, -1, 1))).sum((0, 1)))
    assert np.array_equal(D, (a * a).sum((0, 1)))
    assert np.array_equal(Mg, a.sum((0, 1)))
