"""What the update and training kernels decide or compute without the exact
log and without divisions, compared with them at every input on the device."""
import ctypes

import numpy as np
import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


def test_acclog_screen_exhaustive():
    """thi lies above the correctly rounded log of every one of the 2^23 draws,
    by less than lim (whose last bits the kernels' rounded thi - diff may take),
    and below 0."""
    step = 1 << 21
    for k0 in range(0, 1 << 23, step):
        thi, lim = (x.astype(np.float64) for x in M.acclog_screen_device(k0, step))
        log = M.acclog_host_range(k0, step).astype(np.float64)
        above = thi - log
        assert (above > 0).all() and (above < lim * (1 - 2.0 ** -20)).all() and (thi < 0).all()


def test_silu_of_every_float():
    n, at = ctypes.c_uint64(), ctypes.c_uint32()
    assert M.lib().muca_mlp_silu_check(0, ctypes.byref(n), ctypes.byref(at)) == 0
    assert n.value == 0, (n.value, hex(at.value))
