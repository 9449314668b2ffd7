"""Page-locked host memory: the three planes in one allocation, as a part of a
larger one, and each in an allocation of its own, through uploads, further
passes, both downloads and the quantizer."""
import ctypes

import numpy as np
import pytest

from pik_amd import abi, synth
from pik_amd.devmem import PinnedArray
from pik_amd.runtime import Reconstructor

from .helpers import checker_recon

pytestmark = pytest.mark.gpu


class Planes:
    """Three planes of `shape` in page-locked memory, 7 in every byte around
    and between them."""

    def __init__(self, shape, dtype, layout):
        shape = tuple(shape)
        n = {"one": 3, "part": 5, "apart": 1}[layout]
        first = 1 if layout == "part" else 0
        self.pins = [PinnedArray((n,) + shape, dtype)
                     for _ in range(3 if layout == "apart" else 1)]
        for p in self.pins:
            p.array.view(np.uint8)[...] = 7
        self.views = ([p.array[0] for p in self.pins] if layout == "apart"
                      else [self.pins[0].array[first + c] for c in range(3)])
        self.guards = (self.pins[0].array[::4].view(np.uint8)
                       if layout == "part" else np.zeros(0, np.uint8))

    def fill(self, planes):
        for v, p in zip(self.views, planes):
            v[...] = p
        return self

    def pointers(self):
        return (ctypes.c_void_p * 3)(*[v.ctypes.data for v in self.views])

    def equal(self, want):
        return (all(np.array_equal(v.view(np.uint8), np.ascontiguousarray(
                    w).view(np.uint8)) for v, w in zip(self.views, want)) and
                np.all(self.guards == 7))


# below and above the sizes at which planes are packed or staged together
@pytest.mark.parametrize("w,h", [(61, 47), (520, 264)])
@pytest.mark.parametrize("layout", ["one", "part", "apart"])
def test_decode(w, h, layout):
    fr = synth.make_frame(w, h, seed=w)
    want, _, _ = checker_recon(fr, stages=False)
    ac = Planes(fr.ac.shape[1:], np.int16, layout).fill(fr.ac)
    zero = Planes(fr.ac.shape[1:], np.int16, layout).fill(0 * fr.ac)
    fc, keep = fr.to_c()
    for c in range(3):
        fc.ac[c] = ac.views[c].ctypes.data
    out = Planes((h, w), np.float32, layout)
    with Reconstructor(0) as rec:
        lib, ctx = rec._lib, rec._ctx
        rec._check(lib.pikgpu_frame_upload(ctx, ctypes.byref(fc)))
        rec._check(lib.pikgpu_run(ctx, 0))
        to = ctypes.cast(out.pointers(), ctypes.POINTER(abi.c_float_p * 3))[0]
        rec._check(lib.pikgpu_download(ctx, to, w * 4))
        assert out.equal(want)
        # a pass of zeros adds nothing
        rec._check(lib.pikgpu_frame_add_pass(ctx, zero.pointers(),
                                             fr.ac.shape[2]))
        rec._check(lib.pikgpu_run(ctx, 0))
        for v in out.views:
            v[...] = 3
        rec._check(lib.pikgpu_download(ctx, to, w * 4))
        assert out.equal(want)


@pytest.mark.parametrize("layout", ["one", "part", "apart"])
def test_quantize(layout):
    fr, op = synth.make_opsin_frame(328, 200, seed=4)
    src = Planes(op.shape[1:], np.float32, layout).fill(op)
    ac = Planes(fr.ac.shape[1:], np.int16, layout)
    dc = Planes(fr.dc.shape[1:], np.int16, layout)
    with Reconstructor(0) as rec:
        rec.upload(fr)
        want_ac, want_dc = rec.quantize(op)
        rec.upload(fr)
        rec._check(rec._lib.pikgpu_quantize(
            rec._ctx, src.pointers(), op.shape[2], ac.pointers(),
            fr.ac.shape[2], dc.pointers(), fr.dc.shape[2]))
    assert ac.equal(want_ac) and dc.equal(want_dc)
