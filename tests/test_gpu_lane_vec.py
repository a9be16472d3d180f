"""The lane kernel with several walkers per lane: contexts with enough walkers
for four (phases that end at every word of a Philox block, the smallest L that
loads ahead, FP64 and joint histograms), and batches whose tiles hold two and
four.  Every walker's chain is independent, so sampled walkers are replayed by
the oracle, and E, D, M of all are checked against their lattices."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


def _check(orc, L, W, keying, prec, seed, it, therm, nup, beta, lnw, glat, E, D, Mg, walkers):
    a = glat.reshape(L, L, W).astype(np.int16)
    assert np.array_equal(D, np.abs(a).sum((0, 1))) and np.array_equal(Mg, a.sum((0, 1)))
    assert np.array_equal(E, -(a * (np.roll(a, -1, 0) + np.roll(a, -1, 1))).sum((0, 1)))
    for w in walkers:
        lat = orc.init_lattice(keying, L, 1, seed=seed, w0=w)
        e, d, m = orc.state(L, lat)
        orc.mcs(L, lat, e, d, m, keying=keying, fp64=prec == M.FP64, lnw32=lnw.astype(np.float32),
                lnw64=lnw, iter=it, seed=seed, therm=therm, nupdates=nup, beta=beta, w0=w)
        assert np.array_equal(glat[:, w], lat[0]), w


@pytest.mark.parametrize("L,prec,keying,therm,nup", [
    (10, M.REF32, M.KEYING_WEIGHT, 101, 3), (12, M.FP64, M.KEYING_PRODUCE, 144, 146),
    (16, M.REF32, M.KEYING_WEIGHT, 258, 1), (22, M.REF32, M.KEYING_PRODUCE, 3, 485)])
def test_four_walkers_per_lane(orc, L, prec, keying, therm, nup):
    N, beta, seed = L * L, 1.8, 31
    lnw = -2 * beta * np.arange(N + 1) + np.random.default_rng(L).normal(0, 0.3, N + 1)
    with M.Context(L, 4, precision=prec) as c:
        W = 2048 * c.info.cus - 4
    with M.Context(L, W, beta=beta, precision=prec, keying=keying,
                   joint_blocks=3 if keying == M.KEYING_PRODUCE and prec == M.FP64 else 0,
                   kernel=M.KERNEL_LANE) as ctx:
        ctx.init_lattice(seed=seed)
        ctx.compute_state()
        ctx.set_log_weight(lnw)
        hist, _ = ctx.run(4, seed, therm, nup)
        glat, (E, D, Mg) = ctx.get_lattice(), ctx.get_state()
        if ctx.joint_blocks:   # the joint histogram's sums over M are the D histogram
            j = sum(ctx.get_joint(b) for b in range(3))
            per_d = [j[(d * d + d) // 2:(d * d + d) // 2 + d + 1].sum() for d in range(N + 1)]
            assert np.array_equal(np.array(per_d, np.uint64), hist)
    assert int(hist.sum()) == W * nup
    _check(orc, L, W, keying, prec, seed, 4, therm, nup, beta, lnw, glat, E, D, Mg,
           [0, 1, 2, 3, 1026, W // 2 + 3, W - 1])


def test_batch_with_two_and_four_walkers_per_lane(orc):
    ins = [dict(L=32, walkers=4, seed=7, init_nup=3), dict(L=64, walkers=2052, seed=8),
           dict(L=16, walkers=280000, seed=9, init_nup=5), dict(L=10, walkers=516, seed=10)]
    with M.Batch(ins, tiles=M.KERNEL_LANE) as b:
        b.init(0)
        lnw = [b.get_log_weight(i) for i in range(b.n)]
        b.iterate(1)
        for i, q in enumerate(ins):
            N, W = q["L"] ** 2, q["walkers"]
            nup = q.get("init_nup", 1)
            assert int(b.get_hist(i).sum()) == W * nup
            _check(orc, q["L"], W, M.KEYING_WEIGHT, M.REF32, q["seed"], 0, N, nup, 2.0, lnw[i],
                   b.get_lattice(i), *b.get_state(i), {0, 1, W // 2, W - 1})
