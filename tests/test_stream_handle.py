"""The stream's handle without torch's private call: the public one."""
import importlib.util
import types

import torch


def test_public_call(bws, monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream",
                        lambda index: types.SimpleNamespace(cuda_stream=1000 + index))
    spec = importlib.util.spec_from_file_location("bws_again", bws.__file__)
    m = importlib.util.module_from_spec(spec)
    monkeypatch.setitem(__import__("sys").modules, "bws_again", m)
    spec.loader.exec_module(m)
    assert m._stream() == 1003 and m._stream("cuda:1") == 1001 and m._stream("cuda") == 1003
