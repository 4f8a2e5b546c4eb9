"""Selection of the host extension (csrc/attnres_torch.cpp), without a GPU."""

import os

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


@pytest.mark.skipif(not os.path.exists(H.NATIVE_PATH), reason="the host extension is not built")
def test_available_asks_for_the_extension_too(fresh, monkeypatch, tmp_path):
    assert ops.is_fused_attnres_available()
    monkeypatch.setattr(H, "_native", None)
    monkeypatch.setattr(H, "NATIVE_PATH", str(tmp_path / "missing.so"))
    assert not ops.is_fused_attnres_available()
    other = tmp_path / "other.so"  # (as one built for another torch: the loader refuses it)
    other.write_bytes(b"not a library")
    monkeypatch.setattr(H, "NATIVE_PATH", str(other))
    assert not ops.is_fused_attnres_available()
    monkeypatch.setattr(torch.cuda, "is_available", lambda: False)
    assert not ops.is_fused_attnres_available()
