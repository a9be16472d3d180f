"""The team kernel's layout as the library decides it (no GPU needed)."""
import ctypes

import pytest

import muca_amd as M

LDS = 163840   # bytes per workgroup on an MI355X
NAMES = "eligible lat_lds lds_hist lnw_global rounds order row bytes".split()


def layout(L, W=16, prec=M.REF32, moments=False, cus=256, lds=LDS):
    out = (ctypes.c_uint32 * 8)()
    assert M.lib().muca_test_team_layout(L, W, prec, int(moments), lds, cus, out) == 0
    return dict(zip(NAMES, out))


@pytest.mark.parametrize("cus", [32, 64, 256])
@pytest.mark.parametrize("L,per_cu", [(66, 1), (90, 2), (128, 1)])
def test_moment_windows_start_at_the_resident_walkers_of_the_device(L, per_cu, cus):
    """More walkers than the compute units of this device keep resident, 16 per
    workgroup, read ln W through windows (a partitioned card has fewer units)."""
    W = 16 * per_cu * cus
    at, past = (layout(L, w, M.FP64, True, cus) for w in (W, W + 1))
    assert at["eligible"] and past["eligible"]
    assert LDS // at["bytes"] == per_cu
    assert not at["lnw_global"] and past["lnw_global"] and not past["lat_lds"]
