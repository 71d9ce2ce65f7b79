"""The engine's backward runs on the thread that calls it, whatever the device, and leaves the caller's own setting as it was."""
import threading

import pytest
import torch

from ..common import run_distributed
from ..simple_model import base_config, random_tokens, tiny_llama


def _steps(device, remat, out=None):
    import deepspeedsyclsupport_amd as ds
    from deepspeedsyclsupport_amd.runtime.activation_checkpointing import checkpointing
    eng, _, _, _ = ds.initialize(model=tiny_llama(), config=base_config(stage=1, lr=1e-2, mb=2, clip=1.0))
    seen = []

    def note(grad):
        seen.append((threading.get_ident(), torch._C._is_multithreading_enabled()))

    for x in random_tokens(2, 2, 16, seed=3):
        x = x.to(device)
        loss = eng(x, labels=x)
        loss.register_hook(note)
        if remat:  # a backward inside the backward
            w = torch.randn(4, 4, device=device, requires_grad=True)
            loss = loss + checkpointing.checkpoint(lambda t: (t * t).sum() * 1e-3, w)
            w.register_hook(note)
        eng.backward(loss)
        eng.step()
        assert torch._C._is_multithreading_enabled()
        with torch.autograd.set_multithreading_enabled(False):
            eng.backward(eng(x, labels=x))
            assert not torch._C._is_multithreading_enabled()
        eng.step()
    assert len(seen) == (4 if remat else 2) and set(seen) == {(threading.get_ident(), False)}
    with pytest.raises(RuntimeError):  # (no graph)
        eng.backward(torch.zeros((), device=device))
    assert torch._C._is_multithreading_enabled()


@pytest.mark.parametrize("remat", [False, True])
def test_backward_stays_on_its_thread(remat):
    run_distributed(_steps, 1, "cpu", remat)


@pytest.mark.gpu
@pytest.mark.parametrize("remat", [False, True])
def test_backward_stays_on_its_thread_gpu(remat):
    _steps("cuda", remat)
