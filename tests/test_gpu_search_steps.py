"""The search's own quantization with the forward model, and the sums beside
its steps, against the entry points that do each alone, at sizes around the
tile (32), the colour tile (64) and the 256 blocks of a workgroup."""
import numpy as np
import pytest

from pik_amd import synth
from pik_amd.runtime import Reconstructor
from pik_amd.search import apply_result, search_frame

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(8, 8), (31, 40), (65, 32), (128, 128),
                                 (136, 128), (272, 264)])
@pytest.mark.parametrize("steps", [1, 2])
def test_last_evaluation(w, h, steps):
    fr, opsin, _, lin = synth.make_search_inputs(w, h, seed=w + steps)
    with Reconstructor(0) as rec:
        res = search_frame(rec, fr, opsin, lin, steps=steps)
        final = apply_result(fr, res)
        rec.upload(final)
        ac, dc = rec.quantize(opsin)
        assert np.array_equal(ac, res["ac"]) and np.array_equal(dc, res["dc"])
        field = res["quant_field"].astype(np.float32)
        adj = rec.fwd_adj(field, target=lin)
    # the same partials, summed in the same order
    assert adj["loss"] == res["loss"][-1]
    # the device's float log of each value (at most log(256)) and eight float
    # additions: 2^-21 and 8 x 2^-24 of it
    want = np.log(field.astype(np.float64)).sum()
    assert abs(res["rate"][-1] - want) <= field.size * 5.55 * 2.0 ** -20
