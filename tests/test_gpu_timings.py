"""pikgpu_last_timings: device-clock times per kernel family, for frames with
and without the optional families, within the host's clock around the call."""
import time

import numpy as np
import pytest

from pik_amd import synth
from pik_amd.runtime import Reconstructor

pytestmark = pytest.mark.gpu

RUN = ("dc", "lf_predict", "blocks_idct", "guide", "epf_ar", "dots",
       "final_opsin")


@pytest.mark.parametrize("w,h", [(8, 8), (1030, 520)])
@pytest.mark.parametrize("ar,dots,down", [(1, 3, 1), (1, 0, 1), (0, 0, 1),
                                          (1, 0, 4)])
def test_run_families(w, h, ar, dots, down):
    fr = synth.make_frame(w, h, seed=5, num_dots=dots if w > 64 else 0)
    fr.adaptive_reconstruction = ar
    with Reconstructor(0) as rec:
        assert all(v == 0 for v in rec.timings().values())
        rec.upload(fr)
        rec.set_downsample(down)
        for _ in range(2):
            t0 = time.perf_counter()
            rec.run()
            rec.sync()
            wall = (time.perf_counter() - t0) * 1e3
            t = rec.timings()
            assert all(t[k] >= 0 for k in RUN)
            always = ("dc", "lf_predict", "blocks_idct", "final_opsin")
            assert all(t[k] > 0 for k in always), t
            assert 0 < sum(t[k] for k in RUN) <= wall
            assert (t["guide"] > 0) == bool(ar and down == 1)
            assert (t["epf_ar"] > 0) == (down == 1)
            assert (t["dots"] > 0) == (len(fr.dots) > 0)
            assert t["adj_forward"] == 0 and t["enc_quantize"] == 0


def test_adjoint_and_quantize():
    fr, op = synth.make_opsin_frame(200, 136, seed=6)
    with Reconstructor(0) as rec:
        rec.upload(fr)
        rec.quantize(op)
        assert rec.timings()["enc_quantize"] > 0
        rec.fwd_adj(fr.quant_field.astype(np.float32),
                    target=np.zeros((3, 136, 200), np.float32))
        t = rec.timings()
        assert t["adj_forward"] > 0 and t["adj_backward"] > 0
        assert t["dc"] == 0
