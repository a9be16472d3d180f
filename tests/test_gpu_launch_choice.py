"""A context whose launches go to different kernels (short ones, a
thermalisation with many walkers, production with moments or the joint
histogram) runs the generic kernel's chains."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("obs", [M.OBS_JOINT, M.OBS_MOMENTS])
@pytest.mark.parametrize("L,W", [(16, 40000), (33, 9000), (60, 500)])
def test_mixed_launches(L, W, obs):
    N, B = L * L, 3
    got = []
    for kernel in (M.KERNEL_AUTO, M.KERNEL_GENERIC):
        with M.Context(L, W, beta=1.7, precision=M.FP64, keying=M.KEYING_PRODUCE, joint_blocks=B,
                       observables=obs, kernel=kernel) as ctx:
            ctx.init_lattice(seed=3, stratified=True)
            ctx.compute_state()
            ctx.set_log_weight(-3.5 * np.arange(N + 1.0))
            out = []
            for it, (therm, nup) in enumerate(((N, 0), (0, 1), (0, N // 2 + 3), (3, 2), (N, N // 20))):
                out += [ctx.run(it, 5, therm, nup)[0], *ctx.get_state()]
                if nup:
                    out += [ctx.get_joint(b) if obs == M.OBS_JOINT else
                            np.stack([np.array(x, object) for x in ctx.get_moments(b)])
                            for b in range(B)]
            got.append(out + [ctx.get_lattice()])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
