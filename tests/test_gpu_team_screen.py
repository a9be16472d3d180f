"""FP64 acceptance in the team kernel is screened with FP32 differences of
ln W: whatever ln W holds (steps far above the range of the screen, differences
that overflow FP32, offsets that leave few bits to the differences, equal
neighbours), the chains are the oracle's; lattices and ln W in LDS and in HBM."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu

SHAPES = {
    "rough": lambda r, n: r.normal(0, 40.0, n),
    "huge": lambda r, n: r.choice([-1e300, -1e39, -3.0, 0.0, 2.5, 1e39, 1e300], n),
    "offset": lambda r, n: 1e13 + np.cumsum(r.normal(0, 1.0, n)),
    "flat": lambda r, n: np.zeros(n),
    "steps": lambda r, n: np.cumsum(r.choice([-1.5, 0.0, 1.5], n)),
}


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("L,W,keying", [(24, 35, M.KEYING_WEIGHT), (72, 16, M.KEYING_PRODUCE),
                                        (100, 5, M.KEYING_WEIGHT), (140, 5, M.KEYING_PRODUCE)])
def test_screened_chain_matches_oracle(orc, shape, L, W, keying):
    N, beta, seed = L * L, 1.7, 91
    lnw = SHAPES[shape](np.random.default_rng(L), N + 1)
    lat = orc.init_lattice(keying, L, W, seed=seed, strat_W=W, rounds=7)
    E, D, Mg = orc.state(L, lat)
    with M.Context(L, W, beta=beta, precision=M.FP64, keying=keying) as ctx:
        assert ctx.info.kernel == M.KERNEL_TEAM
        ctx.init_lattice(seed=seed, stratified=True)
        ctx.compute_state()
        ctx.set_log_weight(lnw)
        hist, _ = ctx.run(4, seed, 70, N + 9)
        glat, (gE, gD, gM) = ctx.get_lattice(), ctx.get_state()
    with np.errstate(over="ignore"):
        lnw32 = lnw.astype(np.float32)
    ref = orc.mcs(L, lat, E, D, Mg, keying=keying, fp64=True, rounds=7, lnw32=lnw32, lnw64=lnw,
                  iter=4, seed=seed, therm=70, nupdates=N + 9, beta=beta, nthreads=4)
    assert np.array_equal(hist, ref)
    assert np.array_equal(glat, lat.T)
    assert np.array_equal(gE, E) and np.array_equal(gD, D)
