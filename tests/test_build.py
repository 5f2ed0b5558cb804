"""build.py where torch, or torch's headers, are not installed: what does not need them is still built, without an exception."""
import importlib
import sys

import pytest

builder = importlib.import_module(
    "lancet-accelerating-moe-training-via-whole-graph-computation-communication-overlapping_amd.build")


@pytest.mark.parametrize("missing", ["torch", "headers"])
def test_build_without_torch(monkeypatch, tmp_path, missing):
    if missing == "torch":
        for name in ("torch", "torch.utils", "torch.utils.cpp_extension"):
            monkeypatch.setitem(sys.modules, name, None)
    else:
        from torch.utils import cpp_extension
        monkeypatch.setattr(cpp_extension, "include_paths", lambda *a, **k: [str(tmp_path)])
    monkeypatch.setattr(builder, "build_hip", lambda: "hip")
    monkeypatch.setattr(builder, "build_ops", lambda: "ops")
    monkeypatch.setattr(builder, "_run", lambda cmd: pytest.fail("compiles"))
    assert builder.build_all() == ["hip", "ops"]
