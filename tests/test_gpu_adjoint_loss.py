"""Where pikgpu_fwd_adj leaves the loss with device pointers: the caller's
double, at an 8-byte and at a 4-byte aligned address, with nothing beside it
touched."""
import numpy as np
import pytest

from pik_amd import synth
from pik_amd.devmem import DeviceArray
from pik_amd.runtime import Reconstructor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("at", [0, 1, 2, 3])
def test_loss_address(at):
    w, h = 72, 40
    fr = synth.make_frame(w, h, seed=2)
    qf = fr.quant_field.astype(np.float32)
    target = np.random.default_rng(1).normal(0, 20, (3, h, w)) \
        .astype(np.float32)
    d_loss = DeviceArray.from_numpy(np.full(6, 7, np.float32))
    d_qf, d_target = DeviceArray.from_numpy(qf), DeviceArray.from_numpy(target)
    d_dqf = DeviceArray(qf.shape, np.float32)
    with Reconstructor(0) as rec:
        rec.upload(fr)
        want = rec.fwd_adj(qf, target=target)["loss"]
        rec.fwd_adj_device(d_qf, d_dqf, target=d_target,
                           loss=DeviceArray((1,), np.float64, _base=d_loss,
                                            _ptr=d_loss.data_ptr() + 4 * at))
        rec.sync()
    got = d_loss.numpy()
    assert got[at:at + 2].copy().view(np.float64)[0] == want
    assert np.all(got[:at] == 7) and np.all(got[at + 2:] == 7)
