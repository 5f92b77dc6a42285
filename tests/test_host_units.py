"""Host-side unit tests of device helpers that also compile for the host."""
from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

BIN = Path(__file__).resolve().parent / "cpp" / "_build" / "fastdiv_test"


def test_fastdiv_matches_integer_division():
    if not BIN.exists():
        pytest.skip("tests/cpp not built (run __graft_entry__.build())")
    r = subprocess.run([str(BIN)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "0 wrong" in r.stdout


def test_stream_without_torchs_private_names(monkeypatch):
    """A torch that lacks the raw-stream functions: the current stream through the public ones."""
    import types

    import torch

    from nano_vllm_cpp_amd import ops

    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=77))
    assert ops._make_stream(types.SimpleNamespace())() == 77
