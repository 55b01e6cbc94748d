"""A forked child of a process that has used the GPU must not go on with its
parent's HIP runtime: every entry point is refused, as torch refuses it (CPU)."""
import os

import torch

from lentil_amd import _arrays, _lib


def test_forked_child_asks_torch_again(monkeypatch):
    """The parent's cached device is gone in the child, so torch decides there."""
    monkeypatch.setitem(_lib._devices, 0, torch.device('cuda', 0))     # as after a first call
    monkeypatch.setattr(_lib, '_current_device', lambda: 0)
    monkeypatch.setattr(torch.cuda, 'is_available', lambda: True)

    def refuse():
        raise RuntimeError('Cannot re-initialize CUDA in forked subprocess')
    monkeypatch.setattr(torch.cuda, 'init', refuse)
    assert _lib.device() == torch.device('cuda', 0)

    class Dev(torch.Tensor):
        is_cuda = True
    calls = [_lib.device_index, _lib.device, _lib.context, lambda: _lib.context(torch.device('cuda', 0)),
             lambda: _arrays.is_dev(Dev())]
    pid = os.fork()
    if pid == 0:
        refused = 0
        for call in calls:
            try:
                call()
            except RuntimeError as e:
                refused += 'forked' in str(e)
        os._exit(0 if refused == len(calls) else 1)
    assert os.waitstatus_to_exitcode(os.waitpid(pid, 0)[1]) == 0
    assert _lib.device_index() == 0     # the parent keeps its own
