"""Selection of the host extension (csrc/attnres_torch.cpp), without a GPU."""

import pytest
import torch

import _attnres_hip as H
import attnres_ops as ops


@pytest.fixture
def fresh(monkeypatch):
    """A process that has not used the extension yet, the GPU taken as there."""
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(ops, "_NATIVE", None)
    monkeypatch.setattr(H, "_native", None)


def test_a_traced_call_does_not_load_the_extension(fresh, monkeypatch):
    def native():
        raise AssertionError("loaded while tracing")

    monkeypatch.setattr(H, "native", native)
    monkeypatch.setattr(ops, "_compiling", lambda: True)
    assert ops._native("forward", "backward") is None and ops._NATIVE is None
