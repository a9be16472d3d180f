"""A new context is ready when its constructor returns: what clears its memory
must not run beside the launches that fill it."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


def test_first_lattice_is_not_cleared(orc):
    L, W = 72, 64
    want = orc.init_lattice(M.KEYING_WEIGHT, L, W, seed=7, strat_W=W, rounds=7)
    for _ in range(100):
        with M.Context(L, W, precision=M.FP64) as ctx:
            ctx.init_lattice(seed=7, stratified=True)
            assert np.array_equal(ctx.get_lattice(), want.T)
