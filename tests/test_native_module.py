"""The native call module's own checks when it is set up (no GPU needed)."""

from __future__ import annotations

import pytest
import torch

from vllm_fastdecoder_amd import _lib, build, ops


def test_built_for_this_torch(monkeypatch):
    monkeypatch.setattr(ops, "_NATIVE", None)
    assert ops._native()
    cmd = build.torch_call_command(build.TORCH_CALL_PATH, build.LIB_PATH)
    assert f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}" in cmd


def test_another_torch_is_refused_and_calls_go_through_ctypes(monkeypatch):
    _lib.load_lib()
    from vllm_fastdecoder_amd import _torch_call

    with pytest.raises(ImportError, match="built for torch"):
        _torch_call.init(ops.WORKSPACE.get, ops.device_ptr, None, "1.0.0")
    monkeypatch.setattr(ops, "_NATIVE", None)
    monkeypatch.setattr(torch, "__version__", "1.0.0")
    assert ops._native() is False
