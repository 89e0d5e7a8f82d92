"""The stream that the entry points launch on: torch's current one, with and without torch's private raw-handle function."""
import importlib.util
import types

import pytest
import torch


def _fresh_ops():
    """A copy of catccos_amd.ops of its own, imported now."""
    spec = importlib.util.find_spec("catccos_amd.ops")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_without_the_private_function_the_public_one_answers(monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=4711))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    assert _fresh_ops()._stream() == 4711


@pytest.mark.gpu
def test_both_ways_name_the_current_stream(monkeypatch):
    from catccos_amd import ops
    side = torch.cuda.Stream()
    for _ in range(2):
        assert ops._stream() == torch.cuda.current_stream().cuda_stream
        with torch.cuda.stream(side):
            assert ops._stream() == side.cuda_stream
        monkeypatch.setattr(ops, "_raw_stream", None)
