"""The kernel that MUCA_KERNEL_AUTO takes for one launch (no GPU needed):
thermalisations of production with moments are chosen for as launches without,
and launches too short for the team kernel's set-up go to the others."""
import ctypes

import pytest

import muca_amd as M

T, G, K = M.KERNEL_TEAM, M.KERNEL_GENERIC, M.KERNEL_LANE
LDS, CUS = 163840, 256


def choice(L, W, therm, nup, prec=M.FP64, obs=0, cus=CUS):
    k, b = ctypes.c_int32(), ctypes.c_uint32()
    assert M.lib().muca_test_choose_kernel(L, W, prec, obs, therm, nup, LDS, cus, ctypes.byref(k),
                                           ctypes.byref(b)) == 0
    assert b.value in (64, 128, 256, 512, 1024)
    return k.value


@pytest.mark.parametrize("L,W,therm,nup,kernel", [
    (64, 262144, 4096, 4096, T), (64, 262144, 4096, 0, K), (64, 16384, 4096, 0, T),
    (12, 256016, 144, 49, T), (12, 256016, 144, 0, K), (8, 368496, 64, 22, G),
    (8, 368496, 64, 64, T), (64, 262144, 4096, 256, G), (256, 16384, 65536, 0, T),
    (63, 131072, 3969, 0, G), (63, 131072, 3969, 3969, T)])
def test_moments(L, W, therm, nup, kernel):
    assert choice(L, W, therm, nup, obs=2) == kernel


@pytest.mark.parametrize("L,W,n,kernel", [
    (60, 5279, 1, K), (60, 5279, 3600, T), (67, 1621, 1, G), (67, 1621, 4489, T),
    (100, 4100, 1, K), (100, 4100, 10001, T), (12, 28599, 1, K), (160, 16384, 1, T),
    (36, 65536, 300, K), (36, 65536, 1297, T), (72, 32768, 600, K), (72, 32768, 5184, T)])
def test_short_launches(L, W, n, kernel):
    assert choice(L, W, 0, n) == kernel
    assert choice(L, W, n, 0) == kernel
    assert choice(L, W, n - 1, 1) == kernel


@pytest.mark.parametrize("L", [9, 16, 33, 45, 60, 72, 100, 128, 256])
@pytest.mark.parametrize("W", [1, 16, 4096, 20000])
@pytest.mark.parametrize("obs", [0, 2])
def test_whole_sweeps_stay_on_teams(L, W, obs):
    for therm, nup in ((L * L, 1), (L * L, L * L), (0, L * L)):
        assert choice(L, W, therm, nup, obs=obs) == T
