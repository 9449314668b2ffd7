"""Device functions called by themselves (libpikgpu_check.so)."""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(os.path.join(ROOT, "pik_amd", "libpikgpu_check.so"))


@pytest.mark.parametrize("groups", [1, 512, 513, 4000])
@pytest.mark.parametrize("slow", [0, 3, -1])
def test_end_stamp_is_the_last_waves(lib, groups, slow):
    """The end of a launch is its last wave's, whichever that is: the first
    workgroup's as well as the last one's, and any wave of it."""
    before, stamp = ctypes.c_uint64(), ctypes.c_uint64()
    assert lib.pikgpu_check_stamps(groups, slow % (4 * groups),
                                   ctypes.byref(before),
                                   ctypes.byref(stamp)) == 0
    assert 0 < before.value <= stamp.value


def test_srgb_bytes_of_every_float(lib):
    """The byte is the exact curve's for all 2^32 floats, in each of the three
    places, although the fast value alone would get some wrong; and the window
    in which the exact curve decides is four times their difference."""
    wrong, fast, largest = (ctypes.c_uint64(), ctypes.c_uint64(),
                            ctypes.c_float())
    assert lib.pikgpu_check_srgb(ctypes.byref(wrong), ctypes.byref(fast),
                                 ctypes.byref(largest)) == 0
    print("fast value: %d bytes of 2^32 off, at most %.3g apart"
          % (fast.value, largest.value))
    assert wrong.value == 0
    assert fast.value > 0
    assert 0 < 4 * largest.value < 1 / 4096
