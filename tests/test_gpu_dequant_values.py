"""Dequantisation of every int16 value on the GPU, bit for bit: the decoder
divides 0.145 by the quantized value with a reciprocal and one residual step,
which must give the correctly rounded quotient for each of them."""
import numpy as np
import pytest

from pik_amd import abi, synth
from pik_amd.runtime import Reconstructor

from .helpers import checker_recon

pytestmark = pytest.mark.gpu


def test_every_quantized_value():
    """A frame of DCT8 blocks without predictions whose three AC planes each
    hold all 65536 int16 values: the dequantised coefficients equal the
    oracle's, which divides."""
    fr = synth.make_frame(264, 256, seed=3, predict=False)
    by, bx = fr.ac_strategy.shape
    fr.ac_strategy[...] = abi.ACS_DCT << 4
    rng = np.random.default_rng(1)
    for c in range(3):
        flat = np.zeros((by * bx, 64), np.int16)
        vals = rng.permutation(np.arange(-32768, 32768)).astype(np.int16)
        slots = flat[:, 1:].reshape(-1)[:65536]  # slot 0 is the DC's
        assert slots.size == 65536
        body = np.zeros(by * bx * 63, np.int16)
        body[:65536] = vals
        flat[:, 1:] = body.reshape(-1, 63)
        fr.ac[c] = flat.reshape(by, bx * 64)
        assert len(np.unique(fr.ac[c])) == 65536
    _, want, _ = checker_recon(fr)
    with Reconstructor(0) as rec:
        rec.upload(fr)
        rec.run(keep_stages=True)
        got = rec.stage(abi.STAGE_COEFFS)
    assert np.array_equal(got.view(np.uint32), want["coeffs"].view(np.uint32))
