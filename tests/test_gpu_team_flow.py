"""The team kernel where chunks of whole rounds run on over the ends of rows:
half-rows one and eight attempts longer than whole rounds, FP32 and FP64,
phases that end beside a row's, a half's and a sweep's end, walker counts that
are and are not multiples of 16; against the oracle, production against the
generic kernel, and a batch of one and of several chunk lengths."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,W,prec,keying,rounds", [
    (34, 35, M.REF32, M.KEYING_WEIGHT, 7), (48, 16, M.FP64, M.KEYING_PRODUCE, 7),
    (66, 16, M.REF32, M.KEYING_PRODUCE, 10), (76, 17, M.FP64, M.KEYING_WEIGHT, 7),
    (80, 16, M.REF32, M.KEYING_WEIGHT, 7), (35, 16, M.FP64, M.KEYING_WEIGHT, 10),
    (49, 33, M.REF32, M.KEYING_PRODUCE, 7), (65, 16, M.FP64, M.KEYING_WEIGHT, 7),
    (79, 16, M.REF32, M.KEYING_WEIGHT, 7)])
@pytest.mark.parametrize("therm_off,nup_off", [(0, 1), (-1, 17), (33, -5)])
def test_flowing_chunks_match_oracle(orc, L, W, prec, keying, rounds, therm_off, nup_off):
    N, beta, seed = L * L, 1.6, 78
    therm, nup = N + therm_off, N + N // 2 + nup_off
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


@pytest.mark.parametrize("L", [34, 35])
@pytest.mark.parametrize("observables", [M.OBS_JOINT, M.OBS_MOMENTS])
def test_flowing_production_matches_generic(L, observables):
    W, B = 50, 3
    N = L * L
    got = []
    for kernel in (M.KERNEL_TEAM, M.KERNEL_GENERIC):
        with M.Context(L, W, precision=M.FP64, keying=M.KEYING_PRODUCE, joint_blocks=B,
                       observables=observables, kernel=kernel) as ctx:
            ctx.init_lattice(seed=3, stratified=True)
            ctx.compute_state()
            ctx.set_log_weight(-3.5 * np.arange(N + 1.0))
            h, _ = ctx.run(1, 5, 7, N + 2)
            got.append((h, [ctx.get_joint(b) if observables == M.OBS_JOINT
                            else np.stack([np.array(x, object) for x in ctx.get_moments(b)])
                            for b in range(B)]))
    assert np.array_equal(got[0][0], got[1][0])
    for a, b in zip(got[0][1], got[1][1]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("sizes", [(36, 40, 48), (66, 72), (36, 72, 64, 100, 10)])
def test_flowing_batch_matches_lane_tiles(sizes):
    ins = [dict(L=L, walkers=w, seed=40 + L, init_nup=3, recursion=L != 40, beta=1.5)
           for L, w in zip(sizes, (33, 16, 20, 17, 40))]
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
