"""Walkers whose D is not their lattice's (set from outside, or a lattice set
without computing the state): D would leave [0, N] and with it every table that
is indexed by D, so such walkers run on the generic kernel, which clamps it,
whatever kernel the context has; once the state is computed, or set as the
lattice's, the context's own kernel runs again and gives the oracle's chain."""
import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu

CASES = [(45, 20, M.OBS_JOINT, 0), (45, 20, M.OBS_MOMENTS, 2), (30, 33, M.OBS_MOMENTS, 3),
         (24, 16, M.OBS_JOINT, 2), (72, 5, M.OBS_JOINT, 0), (140, 3, M.OBS_MOMENTS, 1)]


def _run(L, W, obs, blocks, kernel, prepare):
    N = L * L
    with M.Context(L, W, beta=1.7, precision=M.FP64, keying=M.KEYING_PRODUCE, joint_blocks=blocks,
                   observables=obs, kernel=kernel) as ctx:
        prepare(ctx)
        ctx.set_log_weight(-3.4 * np.arange(N + 1.0))
        h, _ = ctx.run(2, 8, 70, N + 5)
        out = [h, ctx.get_lattice(), *ctx.get_state()]
        for b in range(blocks):
            out.append(ctx.get_joint(b) if obs == M.OBS_JOINT
                       else np.stack([np.array(x, object) for x in ctx.get_moments(b)]))
    return out


def _no_state(ctx):
    ctx.init_lattice(seed=5)


def _zero(ctx):
    ctx.init_lattice(seed=5)
    ctx.compute_state()
    ctx.set_state(D=np.zeros(ctx.W))


def _full(ctx):
    ctx.init_lattice(seed=5)
    ctx.compute_state()
    ctx.set_state(D=np.full(ctx.W, ctx.N))


def _one_off(ctx):
    ctx.init_lattice(seed=5)
    ctx.compute_state()
    d = ctx.get_state()[1]
    d[-1] += 1
    ctx.set_state(D=d)


def _lattice_after(ctx):
    ctx.init_lattice(seed=5)
    ctx.compute_state()
    ctx.set_lattice(np.ones((ctx.N, ctx.W)))


@pytest.mark.parametrize("prepare", [_no_state, _zero, _full, _one_off, _lattice_after])
@pytest.mark.parametrize("L,W,obs,blocks", CASES)
def test_foreign_state_runs_as_generic(L, W, obs, blocks, prepare):
    got = _run(L, W, obs, blocks, M.KERNEL_AUTO, prepare)
    ref = _run(L, W, obs, blocks, M.KERNEL_GENERIC, prepare)
    assert got[3].min() >= 0 and got[3].max() <= L * L
    for a, b in zip(got, ref):
        assert np.array_equal(a, b)


def test_lane_kernel():
    for prepare in (_no_state, _zero, _full):
        got = _run(10, 64, M.OBS_JOINT, 1, M.KERNEL_LANE, prepare)
        for a, b in zip(got, _run(10, 64, M.OBS_JOINT, 1, M.KERNEL_GENERIC, prepare)):
            assert np.array_equal(a, b)


def test_autotune_keeps_a_foreign_state_and_every_candidate():
    """Tuned before the state is computed: the choice is made among all kernels
    (4096 walkers: teams by a factor of five) and the walkers are left as they were."""
    with M.Context(64, 4096) as ctx:
        _full(ctx)
        E, _, Mg = ctx.get_state()
        ctx.set_state(E + 1, None, Mg - 1)
        lat, state = ctx.get_lattice(), ctx.get_state()
        ctx.set_log_weight(np.zeros(ctx.N + 1))
        assert ctx.autotune(4000)[0] == M.KERNEL_TEAM
        assert np.array_equal(ctx.get_lattice(), lat)
        for a, b in zip(ctx.get_state(), state):
            assert np.array_equal(a, b)
        ctx.compute_state()
        ctx.run(0, 1, 10, 10)
        D = ctx.get_state()[1]
        assert np.array_equal(D, np.abs(ctx.get_lattice().astype(np.int32)).sum(0))


def test_own_state_set_from_outside(orc):
    L, W, N = 45, 18, 45 * 45
    lnw = -3.4 * np.arange(N + 1.0)
    lat = orc.init_lattice(M.KEYING_WEIGHT, L, W, seed=5, strat_W=W, rounds=7)
    E, D, Mg = orc.state(L, lat)
    with M.Context(L, W, beta=1.7) as ctx:
        ctx.set_lattice(np.zeros((N, W)))
        ctx.set_state(D=np.full(W, 3))
        ctx.set_log_weight(lnw)
        ctx.run(0, 1, 10, 10)
        ctx.set_lattice(lat.T)
        ctx.set_state(E, D, Mg)
        hist, _ = ctx.run(1, 8, 7, N)
        glat, state = ctx.get_lattice(), ctx.get_state()
    ref = orc.mcs(L, lat, E, D, Mg, keying=0, fp64=False, lnw32=lnw.astype(np.float32), lnw64=lnw,
                  iter=1, seed=8, therm=7, nupdates=N, beta=1.7)
    assert np.array_equal(hist, ref) and np.array_equal(glat, lat.T)
    assert np.array_equal(state[0], E) and np.array_equal(state[1], D)
