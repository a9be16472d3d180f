"""ln W with walls (values of an excluded range of D far from the others).  The
float copy of values above 3.4e38 is infinite and the difference of two such is
NaN, which accepts nothing (muca_delta_multigpu.cu:775-782 compares it); in
double, walls cost the rest of the range no time.  The team kernel's chains are
the oracle's, walkers inside and outside the walls; lattices and ln W in LDS
and in HBM, odd L and chunks over row ends."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu

SHAPES = {
    "mixed": lambda r, n: r.choice([-1e300, -1e39, -3.0, 0.0, 2.5, 1e39, 1e300], n),
    "low": lambda r, n: np.where(np.arange(n) % 97 < 60, -1e300, r.normal(0, 1.0, n)),
    "high": lambda r, n: np.where(np.arange(n) % 97 < 60, 1e300, r.normal(0, 1.0, n)),
    # on both sides of the value that decides alone, and of the size whose
    # rounding is left to the exact test
    "near": lambda r, n: np.cumsum(r.choice([-62.0, -61.0, -1.0, 0.5, 61.0, 62.5], n)),
    "far": lambda r, n: np.where(np.arange(n) % 97 < 60, 2.0 ** 33 + r.normal(0, 300.0, n),
                                 r.normal(0, 1.0, n)),
}


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("prec", [M.REF32, M.FP64])
@pytest.mark.parametrize("L,W,keying", [
    (24, 35, M.KEYING_WEIGHT), (30, 16, M.KEYING_PRODUCE), (34, 16, M.KEYING_WEIGHT),
    (45, 20, M.KEYING_WEIGHT), (100, 5, M.KEYING_PRODUCE), (200, 3, M.KEYING_WEIGHT)])
def test_walls_match_oracle(orc, shape, prec, L, W, keying):
    N, beta, seed = L * L, 1.7, 91
    lnw = SHAPES[shape](np.random.default_rng(L), N + 1)
    lat = orc.init_lattice(keying, L, W, seed=seed, strat_W=W, rounds=7)
    E, D, Mg = orc.state(L, lat)
    with M.Context(L, W, beta=beta, precision=prec, keying=keying) as ctx:
        assert ctx.info.kernel == M.KERNEL_TEAM
        ctx.init_lattice(seed=seed, stratified=True)
        ctx.compute_state()
        ctx.set_log_weight(lnw)
        hist, _ = ctx.run(4, seed, 70, N + 9)
        glat, (gE, gD, gM) = ctx.get_lattice(), ctx.get_state()
    with np.errstate(over="ignore"):
        lnw32 = lnw.astype(np.float32)
    ref = orc.mcs(L, lat, E, D, Mg, keying=keying, fp64=prec == M.FP64, rounds=7, lnw32=lnw32,
                  lnw64=lnw, iter=4, seed=seed, therm=70, nupdates=N + 9, beta=beta, nthreads=4)
    assert np.array_equal(hist, ref)
    assert np.array_equal(glat, lat.T)
    assert np.array_equal(gE, E) and np.array_equal(gD, D)


@pytest.mark.parametrize("L,W", [(64, 8192), (72, 4096), (128, 4096)])
@pytest.mark.parametrize("wall", [1e6, -1e6, 1e10, -1e300])
def test_walls_cost_no_time_away_from_them(L, W, wall):
    """One wall below an eighth of the range and one above seven eighths (the
    walkers start at D ~ 2 N / 3): 2.7 times the time when the largest step of
    ln W set the screen's bound for every D; 1.4 allows for the launch's spread."""
    N = L * L
    d = np.arange(N + 1)
    times = {}
    with M.Context(L, W, precision=M.FP64) as ctx:
        for w in (0.0, wall):
            ms = []
            for r in range(4):
                ctx.init_lattice(seed=5)
                ctx.compute_state()
                ctx.set_log_weight(np.where((d < N // 8) | (d > N - N // 8), w, 0.0))
                ms.append(ctx.run(r, 9, N, N // 4, want_hist=False)[1])
            times[w] = min(ms[1:])
    assert times[wall] < 1.4 * times[0.0], times
