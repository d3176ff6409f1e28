"""The plan cache's stream handle, without a GPU: a torch that has no raw-handle function
gives the handle of its Stream object."""
import importlib.util
import types

import torch

from hpxfft_amd import torch_api


def _fresh_torch_api():
    spec = importlib.util.spec_from_file_location("hpxfft_amd.torch_api_fresh", torch_api.__file__)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _streams_of(mod, monkeypatch):
    """The stream each new plan is made with, for the devices 0 and 1."""
    made = []
    monkeypatch.setattr(mod, "Plan", lambda *a, stream, **k: made.append(stream) or stream)

    class Guard:
        def __init__(self, device):
            pass

        def __enter__(self):
            return self

        def __exit__(self, *exc):
            return False

    monkeypatch.setattr(torch.cuda, "device", Guard)
    for i in (0, 1):
        mod._get_plan(8, 8, 1, "f64", 8, 5, torch.device("cuda", i))
    return made


def test_without_the_raw_function(monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: types.SimpleNamespace(cuda_stream=1000 + device))
    assert _streams_of(_fresh_torch_api(), monkeypatch) == [1000, 1001]


def test_with_the_raw_function(monkeypatch):
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 2000 + index, raising=False)
    assert _streams_of(_fresh_torch_api(), monkeypatch) == [2000, 2001]
