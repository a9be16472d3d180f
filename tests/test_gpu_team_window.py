"""The team kernel where D leaves the acceptance window again and again: ln W
so steep that D climbs or falls at almost every step, or random ones, for
every number of rounds per chunk, ragged walker counts and phases that end
inside a round; lattices, E, D, M and the histogram against the oracle."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["up", "down", "random", "ground"])
@pytest.mark.parametrize("L,prec,keying", [
    (8, M.REF32, M.KEYING_WEIGHT), (40, M.FP64, M.KEYING_PRODUCE),
    (72, M.REF32, M.KEYING_WEIGHT), (104, M.REF32, M.KEYING_PRODUCE),
    (136, M.FP64, M.KEYING_WEIGHT), (136, M.FP64, M.KEYING_PRODUCE)])
def test_steep_weights_match_oracle(orc, L, prec, keying, shape):
    N, W, seed, beta = L * L, 19, 4242, 1.7
    rng = np.random.default_rng(L)
    D = np.arange(N + 1)
    lnw = {"up": 20.0 * D, "down": -20.0 * D, "ground": -2 * beta * D,
           "random": rng.normal(0, 3, N + 1)}[shape].astype(np.float64)
    therm, nup = N + 5, 2 * L + 3
    lat = orc.init_lattice(keying, L, W, seed=seed, strat_W=W)
    E, Dd, Mg = orc.state(L, lat)
    with M.Context(L, W, beta=beta, precision=prec, keying=keying, kernel=M.KERNEL_TEAM) as ctx:
        assert ctx.info.kernel == M.KERNEL_TEAM
        ctx.init_lattice(seed=seed, stratified=True)
        ctx.compute_state()
        ctx.set_log_weight(lnw)
        hist, _ = ctx.run(3, seed, therm, nup)
        out = ctx.get_lattice(), *ctx.get_state()
    ref = orc.mcs(L, lat, E, Dd, Mg, keying=keying, fp64=prec == M.FP64,
                  lnw32=lnw.astype(np.float32), lnw64=lnw, iter=3, seed=seed, therm=therm,
                  nupdates=nup, beta=beta)
    assert np.array_equal(hist, ref)
    assert np.array_equal(out[0], lat.T)
    assert np.array_equal(out[1], E) and np.array_equal(out[2], Dd)
    b = out[0].astype(np.int64)
    assert np.array_equal(out[3], b.sum(0))
