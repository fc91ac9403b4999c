"""Host side of the natively issued training step, without a GPU: what the argument block of a step holds."""
import ctypes

import numpy as np
import pytest
import torch

from deepbind_amd import _lib, data, deepity_smat
from deepbind_amd.model import SequenceNet


@pytest.fixture
def no_gpu(monkeypatch):
    """Host tensors taken where the library would refuse them; nothing is launched."""
    for module in (_lib, deepity_smat):
        monkeypatch.setattr(module, "ptr", lambda t: None if t is None else ctypes.c_void_p(t.data_ptr()))
        monkeypatch.setattr(module, "call", lambda name, *args: None)
        monkeypatch.setattr(module, "stream", lambda: None)


def _batch(rng, lens):
    X, R = data.pack_sequences(["ACGT"[i % 4] * n for i, n in enumerate(lens)], 3)
    return torch.from_numpy(X), torch.from_numpy(R), torch.from_numpy(rng.random((len(lens), 1)).astype(np.float32))


def test_input_dropout_changed_between_steps(no_gpu):
    """Every step trains at the rate its net holds when it is issued - on a new batch and on the one before - so that the generator's
    position on the device, which moves by the block's rate, stays where the host's mirror, which moves by the net's, has it."""
    rng = np.random.default_rng(0)
    batches = [_batch(rng, lens) for lens in ([9, 4], [6, 11, 7], [9, 4])]
    net = SequenceNet(1, 4, 4, device="cpu", single_launch=False, dropout=0.5)
    drawn = 0
    for rate, batch in ((0.0, 0), (0.3, 0), (0.3, 1), (0.5, 2), (0.0, 0), (0.0, 1), (0.25, 1), (0.25, 1)):
        net.input_dropout = rate
        X, R, Y = batches[batch]
        net.train_step(X, R, Y)
        a = net._step_args
        assert a.input_rate == np.float32(rate)
        assert rate == 0.0 or (a.Xdrop and a.Mdrop)                # (the step asks for them and they hold the batch)
        assert rate == 0.0 or net._step_buf["Xdrop"].numel() == net._step_buf["Mdrop"].numel() == X.numel()
        drawn += ((X.numel() + 3) // 4 if a.input_rate > 0 else 0) + (R.shape[0] * net.k + 3) // 4
        assert net._rng_offset == drawn
