"""The array for dE/dB where torch finds no memory at first (CPU: torch's allocation is replaced)."""
import pytest
import torch

from psi4_amd import autograd, core


def _failing(monkeypatch, times):
    calls = []
    real = torch.empty

    def empty(*a, **k):
        calls.append("empty")
        if calls.count("empty") <= times:
            raise torch.OutOfMemoryError("out of memory")
        return real(*a, **k)

    monkeypatch.setattr(torch, "empty", empty)
    monkeypatch.setattr(core, "trim_memory", lambda: calls.append("trim"))
    return calls


def test_kept_memory_is_given_back_before_the_second_try(monkeypatch):
    calls = _failing(monkeypatch, 1)
    x = autograd._empty((3, 4, 4), "cpu")
    assert x.shape == (3, 4, 4) and x.dtype == torch.float64
    assert calls == ["empty", "trim", "empty"]


def test_memory_that_is_not_there_is_refused(monkeypatch):
    calls = _failing(monkeypatch, 2)
    with pytest.raises(torch.OutOfMemoryError):
        autograd._empty((3, 4, 4), "cpu")
    assert calls == ["empty", "trim", "empty"]


def test_nothing_is_given_back_without_need(monkeypatch):
    calls = _failing(monkeypatch, 0)
    autograd._empty((2, 2, 2), "cpu")
    assert calls == ["empty"]
