"""The lane kernel with four walkers per lane, where test_gpu_lane_vec.py does
not go: the joint histogram bin by bin, the D histogram in HBM, the carry of a
wrapped LDS bin, and batches in double with two and four walkers per lane and
an instance whose histogram does not fit in LDS."""
import numpy as np
import pytest

import muca_amd as M
from test_gpu_lane_vec import _check

pytestmark = pytest.mark.gpu


def _walkers(extra):
    with M.Context(10, 4) as c:
        return 1536 * c.info.cus + extra   # the fewest that take four per lane


def _run(L, W, kernel, therm, nup, blocks=0, preload=0, prec=M.FP64, keying=M.KEYING_PRODUCE):
    N = L * L
    lnw = -3.4 * np.arange(N + 1) + np.random.default_rng(L).normal(0, 0.3, N + 1)
    with M.Context(L, W, beta=1.7, precision=prec, keying=keying, joint_blocks=blocks,
                   kernel=kernel) as ctx:
        ctx.set_test_hist_preload(preload)
        ctx.init_lattice(seed=12)
        ctx.compute_state()
        ctx.set_log_weight(lnw)
        h, _ = ctx.run(3, 6, therm, nup)
        return [h, *ctx.get_state()] + [ctx.get_joint(b) for b in range(blocks)]


@pytest.mark.parametrize("L,therm,nup,blocks", [(10, 31, 135, 3), (24, 0, 577, 1), (34, 5, 66, 5)])
def test_joint_histogram_bin_by_bin(L, therm, nup, blocks):
    W = _walkers(28)
    for a, b in zip(_run(L, W, M.KERNEL_LANE, therm, nup, blocks),
                    _run(L, W, M.KERNEL_GENERIC, therm, nup, blocks)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("L", [118, 142])
def test_histogram_in_hbm(L):
    W = _walkers(4)
    for a, b in zip(_run(L, W, M.KERNEL_LANE, 6, 37), _run(L, W, M.KERNEL_GENERIC, 6, 37)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("prec,keying", [(M.REF32, M.KEYING_WEIGHT), (M.FP64, M.KEYING_PRODUCE)])
def test_wrapped_bins_carry(prec, keying):
    W = _walkers(12)
    kw = dict(therm=2, nup=259, prec=prec, keying=keying)
    plain = _run(12, W, M.KERNEL_LANE, **kw)
    wrapped = _run(12, W, M.KERNEL_LANE, preload=0xFFFFFFF0, **kw)
    assert int(plain[0].sum()) == W * 259
    for a, b in zip(plain, wrapped):
        assert np.array_equal(a, b)


def test_batch_in_double_with_two_and_four_walkers_per_lane(orc):
    ins = [dict(L=32, walkers=4, seed=7, init_nup=3), dict(L=64, walkers=2052, seed=8),
           dict(L=16, walkers=280000, seed=9, init_nup=5), dict(L=10, walkers=516, seed=10),
           dict(L=118, walkers=520, seed=11, init_nup=2)]
    with M.Batch(ins, tiles=M.KERNEL_LANE, precision=M.FP64) as b:
        b.init(0)
        lnw = [b.get_log_weight(i) for i in range(b.n)]
        b.iterate(1)
        for i, q in enumerate(ins):
            N, W = q["L"] ** 2, q["walkers"]
            nup = q.get("init_nup", 1)
            assert int(b.get_hist(i).sum()) == W * nup
            _check(orc, q["L"], W, M.KEYING_WEIGHT, M.FP64, q["seed"], 0, N, nup, 2.0, lnw[i],
                   b.get_lattice(i), *b.get_state(i), {0, 1, W // 2, W - 1})
