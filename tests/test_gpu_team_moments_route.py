"""Production with per-D moments and more walkers than lattices in LDS keep
resident: ln W windows and lattices from HBM, against the generic kernel, on
both sides of the line and for walker counts that are no multiple of 16."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,W", [(50, 12290), (66, 4096), (66, 4100), (90, 8200)])
def test_moments_match_generic(L, W):
    N, B = L * L, 2
    lnw = -3.5 * np.arange(N + 1.0) + np.random.default_rng(L).normal(0, 0.3, N + 1)
    got = []
    for kernel in (M.KERNEL_TEAM, M.KERNEL_GENERIC):
        with M.Context(L, W, beta=1.7, precision=M.FP64, keying=M.KEYING_PRODUCE, joint_blocks=B,
                       observables=M.OBS_MOMENTS, kernel=kernel) as ctx:
            ctx.init_lattice(seed=3, stratified=True)
            ctx.compute_state()
            ctx.set_log_weight(lnw)
            h, _ = ctx.run(1, 5, 7, 333)
            got.append([h, ctx.get_lattice(), *ctx.get_state()] +
                       [np.stack([np.array(x, object) for x in ctx.get_moments(b)])
                        for b in range(B)])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
