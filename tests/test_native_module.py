"""The extension module of the layer calls reads tensors' fields where the torch it was built against has them: with any other it must
not be used."""
import pytest
import torch


def test_module_of_another_torch_is_refused(sb, monkeypatch):
    assert sb._native.calls().torch_version == torch.__version__
    monkeypatch.setattr(sb._native, "_calls_module", None)
    monkeypatch.setattr(torch, "__version__", "1.0.0")
    with pytest.raises(sb._native.NativeLibraryError, match="1.0.0"):
        sb._native.calls()
    assert sb._native._calls_module is None
