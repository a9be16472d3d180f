"""The lane kernel's launch shape (no GPU needed): a workgroup has the lanes
that were asked for, so that a context reports what it runs and the autotuner's
candidates are different launches."""
import ctypes

import pytest

import muca_amd as M


def _shape(L, W, block, cus=256):
    lanes, per = ctypes.c_uint32(), ctypes.c_uint32()
    assert M.lib().muca_test_lane_shape(L, W, cus, block, ctypes.byref(lanes),
                                        ctypes.byref(per)) == 0
    return lanes.value, per.value


@pytest.mark.parametrize("block", [64, 128, 256, 512, 1024])
@pytest.mark.parametrize("L,W", [(72, 524288), (10, 393216), (72, 4096), (8, 524288), (72, 393214)])
def test_workgroups_have_the_lanes_asked_for(L, W, block):
    lanes, per = _shape(L, W, block)
    assert lanes == block
    assert per == (4 if L > 8 and W % 4 == 0 and W >= 1536 * 256 and block <= 512 else 1)


def test_autotune_candidates_differ():
    for L, W in ((72, 524288), (72, 4096)):
        assert len({_shape(L, W, b) for b in (256, 512, 1024)}) == 3
