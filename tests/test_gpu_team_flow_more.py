"""Chunks over row ends where half-rows are two rounds and seven or eight
attempts long: L = 78, and L = 80 where no histogram shares LDS with the
lattices (with one, L = 80 keeps them in HBM and works row by row)."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,keying", [(M.REF32, M.KEYING_WEIGHT), (M.FP64, M.KEYING_PRODUCE)])
def test_seven_attempts_over(orc, prec, keying):
    L, W, beta, seed = 78, 18, 1.6, 44
    N = L * L
    lnw = -2 * beta * np.arange(N + 1) + np.random.default_rng(L).normal(0, 0.3, N + 1)
    lat = orc.init_lattice(keying, L, W, seed=seed, strat_W=W, rounds=7)
    E, D, Mg = orc.state(L, lat)
    with M.Context(L, W, beta=beta, precision=prec, keying=keying) as ctx:
        assert ctx.info.kernel == M.KERNEL_TEAM and ctx.info.lds_lattice == 1
        ctx.init_lattice(seed=seed, stratified=True)
        ctx.compute_state()
        ctx.set_log_weight(lnw)
        hist, _ = ctx.run(9, seed, N + 33, N + N // 2 - 5)
        glat = ctx.get_lattice()
    ref = orc.mcs(L, lat, E, D, Mg, keying=keying, fp64=prec == M.FP64,
                  lnw32=lnw.astype(np.float32), lnw64=lnw, iter=9, seed=seed, therm=N + 33,
                  nupdates=N + N // 2 - 5, beta=beta, nthreads=4)
    assert np.array_equal(hist, ref) and np.array_equal(glat, lat.T)


def test_eight_attempts_over():
    L, W, B = 80, 35, 2
    N = L * L
    got = []
    for kernel in (M.KERNEL_AUTO, M.KERNEL_GENERIC):
        with M.Context(L, W, beta=1.7, precision=M.FP64, keying=M.KEYING_PRODUCE, joint_blocks=B,
                       observables=M.OBS_MOMENTS, kernel=kernel) as ctx:
            if kernel == M.KERNEL_AUTO:
                assert ctx.info.kernel == M.KERNEL_TEAM and ctx.info.lds_lattice == 1
            ctx.init_lattice(seed=3, stratified=True)
            ctx.compute_state()
            ctx.set_log_weight(-3.5 * np.arange(N + 1.0))
            h, _ = ctx.run(1, 5, 7, N + 41)
            got.append([h, ctx.get_lattice(), *ctx.get_state()] +
                       [np.stack([np.array(x, object) for x in ctx.get_moments(b)])
                        for b in range(B)])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
