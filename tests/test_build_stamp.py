"""The build stamps: the HIP library's over its sources, the autograd node's over its own source and what it is compiled
against."""
import pytest
import torch

from pymolecular_amd import _build, _capi


def test_node_stamp_follows_what_it_is_compiled_against(monkeypatch):
    base, lib = _build.ext_hash(), _build.source_hash()
    assert _build.EXT_STAMP.read_text().strip() == base
    for change in (lambda m: m.setattr(torch, "__version__", "0.0"),
                   lambda m: m.setattr(torch, "compiled_with_cxx11_abi", lambda: "other"),
                   lambda m: m.setattr(_build, "EXT_FLAGS", _build.EXT_FLAGS + ["-O0"])):
        with monkeypatch.context() as m:
            change(m)
            assert _build.ext_hash() != base and _build.source_hash() == lib


@pytest.mark.parametrize("what", ["torch", "stamp", "module"])
def test_foreign_node_is_refused(what, monkeypatch, tmp_path):
    monkeypatch.setattr(_capi, "_ext", None)
    if what == "torch":
        monkeypatch.setattr(torch, "__version__", "0.0")
    elif what == "stamp":
        monkeypatch.setattr(_build, "EXT_STAMP", tmp_path / "none.srchash")
    else:
        monkeypatch.setattr(_build, "EXT", tmp_path / "none.so")
    with pytest.raises(RuntimeError, match="_build"):
        _capi.ext()
    monkeypatch.undo()
    assert _capi.ext() is not None
