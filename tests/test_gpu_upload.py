"""Uploads on both sides of each of their rules: AC planes packed with the
rest of the frame (up to 256 KB, 682 blocks) or copied on their own, rows with
a pitch of their own, a frame's other inputs above the staging buffer (16 MB),
and what an upload leaves to the next call."""
import numpy as np
import pytest

from pik_amd import synth
from pik_amd.runtime import PikGpuError, Reconstructor

from .helpers import checker_recon

pytestmark = pytest.mark.gpu


def padded(a, extra):
    """A copy of `a` whose rows have `extra` unused entries behind them."""
    wide = np.full(a.shape[:-1] + (a.shape[-1] + extra,), 77, a.dtype)
    wide[..., :a.shape[-1]] = a
    return wide[..., :a.shape[-1]]


def same(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("w,h", [(8, 8), (176, 248), (8, 5464), (520, 264)])
@pytest.mark.parametrize("pad", [False, True])
def test_decode_matches_oracle(w, h, pad):
    fr = synth.make_frame(w, h, seed=w + h, lut_ids="rand",
                          num_dots=2 if w > 64 else 0)
    want, _, _ = checker_recon(fr, stages=False)
    if pad:
        for i, name in enumerate(("ac", "dc", "quant_field", "ac_strategy",
                                  "sigma_lut_ids", "dequant_cf", "ytox_map",
                                  "ytob_map")):
            setattr(fr, name, padded(getattr(fr, name), 1 + i))
    with Reconstructor(0) as rec:
        assert same(rec.reconstruct(fr), want)


def test_large_side_inputs():
    fr = synth.make_frame(72, 40, seed=3)
    want, _, _ = checker_recon(fr, stages=False)
    table = np.ones((17 << 20) // 4, np.float32)
    table[:fr.dequant_table.size] = fr.dequant_table
    fr.dequant_table = table
    with Reconstructor(0) as rec:
        assert same(rec.reconstruct(fr), want)


def test_large_side_inputs_with_dots():
    """The dots' tile lists go from host memory of the library's own."""
    fr = synth.make_frame(520, 264, seed=3, num_dots=40)
    want, _, _ = checker_recon(fr, stages=False)
    table = np.ones((17 << 20) // 4, np.float32)
    table[:fr.dequant_table.size] = fr.dequant_table
    fr.dequant_table = table
    with Reconstructor(0) as rec:
        assert same(rec.reconstruct(fr), want)


def test_refused_frame_between_two():
    good = synth.make_frame(320, 200, seed=1)
    bad = synth.make_frame(320, 200, seed=2)
    bad.quant_field = bad.quant_field.copy()
    bad.quant_field[0, 0] = -1
    with Reconstructor(0) as rec:
        want = rec.reconstruct(good)
        with pytest.raises(PikGpuError):
            rec.upload(bad)
        assert same(rec.reconstruct(good), want)


def test_quantize_uses_the_uploaded_table():
    fr, op = synth.make_opsin_frame(120, 72, seed=4)
    other, _ = synth.make_opsin_frame(120, 72, seed=4)
    other.dequant_table = other.dequant_table * np.float32(1.5)

    def quantized(rec, f):
        rec.upload(f)
        return rec.quantize(op)

    with Reconstructor(0) as a, Reconstructor(0) as b:
        quantized(a, fr)
        got, want = quantized(a, other), quantized(b, other)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
