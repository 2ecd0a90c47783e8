"""The stream of a call that names none: torch's current stream, read through
private functions of torch where it has them and through the public call where
not. A failure there is never a launch on the null stream. No GPU needed: torch
is stood in for."""
import types

import pytest
import torch

import smallaios_amd as S

RAW = "_cuda_getCurrentRawStream"


def stand_in(monkeypatch, *, raw=None, public=None, available=True, missing=()):
    """torch.cuda initialised; its stream functions replaced."""
    def current_stream():
        if isinstance(public, Exception):
            raise public
        return types.SimpleNamespace(cuda_stream=public)

    monkeypatch.setattr(S, "_torch_state", None)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(torch.cuda, "is_available", lambda: available)
    monkeypatch.setattr(torch.cuda, "current_stream", current_stream)
    monkeypatch.setattr(torch._C, RAW, raw or (lambda device: 77 + device), raising=False)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 3, raising=False)
    for name in missing:
        monkeypatch.delattr(torch._C, name)


def test_current_stream_is_read_as_a_number(monkeypatch):
    stand_in(monkeypatch, public=1234)
    assert S._stream(None) == 80
    assert S._stream(5) == 5
    assert S._stream(types.SimpleNamespace(cuda_stream=6)) == 6


@pytest.mark.parametrize("missing", [(RAW,), ("_cuda_getDevice",), (RAW, "_cuda_getDevice")])
def test_public_call_where_torch_lacks_the_private_ones(monkeypatch, missing):
    stand_in(monkeypatch, public=1234, missing=missing)
    assert S._stream(None) == 1234


def test_public_call_before_initialisation(monkeypatch):
    stand_in(monkeypatch, public=1234)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: False)
    assert S._stream(None) == 1234


def test_failures_are_raised(monkeypatch):
    def changed(device):
        raise TypeError("another signature")

    stand_in(monkeypatch, raw=changed, public=1234)
    with pytest.raises(TypeError):
        S._stream(None)
    stand_in(monkeypatch, public=RuntimeError("device lost"), missing=(RAW,))
    with pytest.raises(RuntimeError):
        S._stream(None)


def test_torch_without_a_gpu_has_no_current_stream(monkeypatch):
    stand_in(monkeypatch, public=RuntimeError("no GPU"), available=False, missing=(RAW,))
    assert S._stream(None) is None
