"""The batch kernels' static LDS is within what their launches leave free."""
import ctypes

import pytest

import muca_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [M.REF32, M.FP64])
@pytest.mark.parametrize("tiles,several", [(M.KERNEL_TEAM, 0), (M.KERNEL_LANE, 0),
                                           (M.KERNEL_LANE, 1)])
def test_static_lds_is_reserved(prec, tiles, several):
    used, kept = ctypes.c_uint32(), ctypes.c_uint32()
    assert M.lib().muca_test_batch_static_lds(prec, tiles, several, ctypes.byref(used),
                                              ctypes.byref(kept)) == 0
    assert 0 < used.value <= kept.value
