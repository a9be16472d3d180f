"""E, D and M of every instance of a batch, computed in one launch: sizes and
walker counts of different remainders side by side, against the oracle."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("walkers", [(128, 129, 4, 1, 260), (64, 64, 64, 64, 64)])
def test_batch_state_matches_oracle(orc, walkers):
    sizes = (8, 24, 34, 64, 10)
    with M.Batch([dict(L=L, walkers=w, seed=7 + L, beta=1.5) for L, w in zip(sizes, walkers)]) as b:
        for _ in range(2):
            b.init(0)
            for i, L in enumerate(sizes):
                lat = b.get_lattice(i)
                E, D, Mg = orc.state(L, np.ascontiguousarray(lat.T))
                got = b.get_state(i)
                assert all(np.array_equal(x, y) for x, y in zip(got, (E, D, Mg)))
            b.iterate(1)
