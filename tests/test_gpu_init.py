"""Initial lattices, four walkers per thread or one, against the oracle: odd
lattices whose last Philox block is part used, walker counts that are and are
not multiples of four, both starts and keyings."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stratified", [False, True])
@pytest.mark.parametrize("keying", [M.KEYING_WEIGHT, M.KEYING_PRODUCE])
@pytest.mark.parametrize("L,W,rounds", [(2, 4, 7), (5, 1028, 7), (33, 4, 10), (33, 77, 7),
                                        (40, 260, 10)])
def test_init_matches_oracle(orc, keying, L, W, rounds, stratified):
    with M.Context(L, W, keying=keying, rounds=rounds) as ctx:
        ctx.init_lattice(mm=3, gpu=1, seed=4321, stratified=stratified)
        lat = ctx.get_lattice()
    ref = orc.init_lattice(keying, L, W, mm=3, gpu=1, seed=4321, rounds=rounds,
                           strat_W=W if stratified else 0)
    assert np.array_equal(lat, ref.T)
