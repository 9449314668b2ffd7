"""Decodes at the sizes where the launch chain changes shape: the smallest
images (every edge of the mirrored guide border in one tile), the largest and
the next number of min/max partials that the guide kernel reduces itself (512
and 513 row ranges of 8), DC images of one and of several of their filter's
tiles (32 x 8 blocks), the last row of 2, 4, 8 and 16 per workgroup of the final
kernel and of 2, 3 and more per range of the min/max kernel, and more blocks than one pass of the DC kernel's 256
workgroups takes (65536)."""
import numpy as np
import pytest

from pik_amd import synth
from pik_amd.runtime import BatchReconstructor, Reconstructor

from .helpers import checker_recon

pytestmark = pytest.mark.gpu

SIZES = [(8, 8), (16, 8), (8, 24), (13, 31), (37, 33), (64, 40), (256, 64),
         (264, 72), (248, 520), (40, 1030), (505, 2043), (1277, 1637),
         (40, 4096), (40, 4097), (2049, 2048)]


@pytest.fixture(scope="module")
def rec():
    with Reconstructor(0) as r:
        yield r


@pytest.mark.parametrize("w,h", SIZES)
def test_decode_matches_oracle(rec, w, h):
    fr = synth.make_frame(w, h, seed=w * 3 + h, lut_ids="rand")
    want, _, _ = checker_recon(fr, stages=False)
    got = rec.reconstruct(fr)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_batch_of_the_same_sizes(rec):
    frames = [synth.make_frame(w, h, seed=w * 3 + h) for w, h in SIZES]
    with BatchReconstructor(0) as b:
        got = b.reconstruct(frames)
    for fr, g in zip(frames, got):
        want = rec.reconstruct(fr)
        assert np.array_equal(g.view(np.uint32), want.view(np.uint32)), \
            (fr.xsize, fr.ysize)
