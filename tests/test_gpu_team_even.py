"""The team kernel at even L that are no multiple of 8, where a half-row is
not a whole number of Philox blocks: phases that end at every word of a block,
half-rows of one or two chunks, lattices and ln W in LDS or in HBM, against
the oracle; and a batch of such lattices against lane tiles."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,prec,keying,rounds", [
    (10, M.REF32, M.KEYING_WEIGHT, 7), (12, M.FP64, M.KEYING_PRODUCE, 10),
    (18, M.FP64, M.KEYING_WEIGHT, 7), (34, M.REF32, M.KEYING_PRODUCE, 7),
    (50, M.REF32, M.KEYING_WEIGHT, 10), (70, M.FP64, M.KEYING_PRODUCE, 7),
    (100, M.REF32, M.KEYING_WEIGHT, 7), (130, M.REF32, M.KEYING_WEIGHT, 7),
    (138, M.FP64, M.KEYING_PRODUCE, 7), (254, M.FP64, M.KEYING_WEIGHT, 7)])
@pytest.mark.parametrize("therm_off,nup_off", [(-3, 1), (2, -1), (-1, 6)])
def test_even_sizes_match_oracle(orc, L, prec, keying, rounds, therm_off, nup_off):
    N, W, beta, seed = L * L, 5 if L > 100 else 35, 1.6, 77
    therm, nup = N // 2 + L // 2 + therm_off, L + nup_off if L > 200 else N + nup_off
    lnw = -2 * beta * np.arange(N + 1) + np.random.default_rng(L).normal(0, 0.3, N + 1)
    lat = orc.init_lattice(keying, L, W, seed=seed, strat_W=W, rounds=rounds)
    E, D, Mg = orc.state(L, lat)
    with M.Context(L, W, beta=beta, precision=prec, keying=keying, rounds=rounds) as ctx:
        assert ctx.info.kernel == M.KERNEL_TEAM
        ctx.init_lattice(seed=seed, stratified=True)
        ctx.compute_state()
        ctx.set_log_weight(lnw)
        hist, _ = ctx.run(9, seed, therm, nup)
        glat, (gE, gD, gM) = ctx.get_lattice(), ctx.get_state()
    ref = orc.mcs(L, lat, E, D, Mg, keying=keying, fp64=prec == M.FP64, rounds=rounds,
                  lnw32=lnw.astype(np.float32), lnw64=lnw, iter=9, seed=seed, therm=therm,
                  nupdates=nup, beta=beta, nthreads=4)
    assert np.array_equal(hist, ref)
    assert np.array_equal(glat, lat.T)
    assert np.array_equal(gE, E) and np.array_equal(gD, D)
    assert np.array_equal(gM, glat.astype(np.int64).sum(0))


@pytest.mark.parametrize("observables", [M.OBS_JOINT, M.OBS_MOMENTS])
def test_even_production_matches_generic(observables):
    L, W, B = 22, 50, 3
    N = L * L
    lnw = -3.5 * np.arange(N + 1.0)
    got = []
    for kernel in (M.KERNEL_TEAM, M.KERNEL_GENERIC):
        with M.Context(L, W, precision=M.FP64, keying=M.KEYING_PRODUCE, joint_blocks=B,
                       observables=observables, kernel=kernel) as ctx:
            ctx.init_lattice(seed=3, stratified=True)
            ctx.compute_state()
            ctx.set_log_weight(lnw)
            h, _ = ctx.run(1, 5, 7, N + 2)
            got.append((h, [ctx.get_joint(b) if observables == M.OBS_JOINT
                            else np.stack([np.array(x, object) for x in ctx.get_moments(b)])
                            for b in range(B)]))
    assert np.array_equal(got[0][0], got[1][0])
    for a, b in zip(got[0][1], got[1][1]):
        assert np.array_equal(a, b)


def test_even_batch_matches_lane_tiles():
    ins = [dict(L=L, walkers=w, seed=40 + L, init_nup=nup, recursion=r, beta=1.5)
           for L, w, nup, r in ((10, 33, 5, True), (18, 16, 7, False), (50, 20, 3, True),
                                (100, 17, 2, False), (24, 40, 1, True))]
    got = []
    for tiles in (M.KERNEL_AUTO, M.KERNEL_LANE):
        with M.Batch(ins, tiles=tiles) as b:
            assert b.tiles == (M.KERNEL_TEAM if tiles == M.KERNEL_AUTO else M.KERNEL_LANE)
            b.init(0)
            b.iterate(9)
            got.append([(b.get_hist(i), b.get_log_weight(i), b.get_lattice(i))
                        for i in range(b.n)])
    for x, y in zip(*got):
        assert all(np.array_equal(p, q) for p, q in zip(x, y))
