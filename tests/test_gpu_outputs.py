"""Downloads over every route the library takes from its dense output rows to
host memory: one linear copy, small planes staged together, short strided
rows through staging, long strided rows as a 2-D copy; widths that are no
multiple of 4 and images at and past the staging limits."""
import ctypes

import numpy as np
import pytest

from pik_amd import abi, synth
from pik_amd.runtime import Reconstructor

from .helpers import checker_recon
from .srgb import srgb8

pytestmark = pytest.mark.gpu

# (width, height): below, at and above 128 KB of output planes; rows of
# 32 KB (8192 floats) and more
SIZES = [(9, 8), (61, 47), (104, 105), (105, 104), (203, 131), (8190, 16),
         (8195, 9)]


@pytest.fixture(scope="module")
def rec():
    with Reconstructor(0) as r:
        yield r


def _strided(shape, row, dtype):
    """An array of `shape` whose rows lie `row` elements apart, guards set."""
    base = np.full(shape[:-1] + (row,), 7, dtype)
    return base, base[..., :shape[-1]]


@pytest.mark.parametrize("w,h", SIZES)
def test_linear_and_srgb8_downloads(rec, w, h):
    frame = synth.make_frame(w, h, seed=w + h)
    want, _, _ = checker_recon(frame, stages=False)
    bytes_ = srgb8(want).transpose(1, 2, 0)
    rec.upload(frame)
    rec.set_output(abi.OUTPUT_LINEAR | abi.OUTPUT_SRGB8)
    rec.run()
    rec.set_output(abi.OUTPUT_LINEAR)
    for pad in (0, 1, 33):
        base, out = _strided((3, h, w), w + pad, np.float32)
        rec.download(out=out)
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32)), pad
        assert np.all(base[..., w:] == 7)
        base, out = _strided((h, 3 * w), 3 * w + pad, np.uint8)
        rec._check(rec._lib.pikgpu_download_srgb8(
            rec._ctx, ctypes.c_void_p(base.ctypes.data), 3 * w + pad))
        # the transfer function in float32 differs from float64 only where
        # the value lies within float32 rounding of the next byte
        diff = np.abs(out.reshape(h, w, 3).astype(np.int32) - bytes_)
        assert diff.max() <= 1 and (diff != 0).mean() < 1e-3, pad
        assert np.all(base[..., 3 * w:] == 7)


@pytest.mark.parametrize("w,h", [(105, 104), (203, 131), (203, 132)])
def test_planes_one_by_one(rec, w, h):
    """Dense host planes behind one another, apart, and in another order."""
    frame = synth.make_frame(w, h, seed=w + h)
    want, _, _ = checker_recon(frame, stages=False)
    rec.upload(frame)
    rec.run()
    for order in ((0, 1, 2), (2, 1, 0), (0, 2, 4), (0, 1, 3)):
        base = np.full((5, h, w), 7, np.float32)
        planes = (abi.c_float_p * 3)(
            *[base[i].ctypes.data_as(abi.c_float_p) for i in order])
        rec._check(rec._lib.pikgpu_download(rec._ctx, planes, w * 4))
        for c, i in enumerate(order):
            assert np.array_equal(base[i].view(np.uint32),
                                  want[c].view(np.uint32)), order
        for i in set(range(5)) - set(order):
            assert np.all(base[i] == 7), order
