"""How calls choose between the native extension and the general path (no GPU)."""
import sys
import warnings

import pytest
import torch  # noqa: F401  (the extension is asked for only where PyTorch is loaded)

import tensorcomprehensions_amd as tc


class _Uncalled:
    _native = None


def test_a_missing_extension_is_reported_once(monkeypatch):
    monkeypatch.setitem(sys.modules, "tensorcomprehensions_amd._torch_call", None)
    monkeypatch.setattr(tc, "_reported", False)
    with pytest.warns(RuntimeWarning, match="general path"):
        first = _Uncalled()
        assert tc._plan(first).run([], []) is False and first._native is tc._NO_PLAN
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert tc._plan(_Uncalled()).call([]) is None
