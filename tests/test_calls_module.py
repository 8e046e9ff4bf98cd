"""The native calls (csrc/bind.cpp) are optional: without a module that loads, and that was built for this interpreter and this torch, fused.py makes
the calls itself, and the library builds without it."""
import os
import shutil
import subprocess
import warnings

import pytest

from llvq_amd import _ffi


@pytest.fixture()
def asked_anew(monkeypatch):
    pytest.importorskip("torch")
    monkeypatch.setattr(_ffi, "_calls", _ffi._NOT_ASKED)
    return monkeypatch


def _refused(match):
    with pytest.warns(RuntimeWarning, match=match):
        assert _ffi.calls() is None
    with warnings.catch_warnings():  # said once
        warnings.simplefilter("error")
        assert _ffi.calls() is None


def test_a_module_that_does_not_load_is_not_used(asked_anew, tmp_path):
    for name, data in (("empty.so", b""), ("cut.so", b"\x7fELF\x02\x01\x01" + bytes(9))):
        (tmp_path / name).write_bytes(data)
        asked_anew.setattr(_ffi, "_CALLS", str(tmp_path / name))
        asked_anew.setattr(_ffi, "_calls", _ffi._NOT_ASKED)
        _refused("is not used")


@pytest.mark.skipif(not os.path.exists(_ffi._CALLS), reason="csrc/bind.cpp was not built")
def test_a_module_of_another_build_is_not_used(asked_anew):
    module = _ffi.calls()
    assert module is not None and module.built_for == _ffi._built_for()
    asked_anew.setattr(_ffi, "_calls", _ffi._NOT_ASKED)
    asked_anew.setattr(_ffi, "_built_for", lambda: "1.0.0/cpython-30")
    _refused("it was built for")


def test_no_module_is_no_error(asked_anew, tmp_path):
    asked_anew.setattr(_ffi, "_CALLS", str(tmp_path / "none.so"))
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _ffi.calls() is None


def test_the_build_goes_on_without_it(monkeypatch, tmp_path, capsys):
    """...and leaves no older one behind."""
    import __graft_entry__ as entry

    if not os.path.exists(_ffi._LIB):
        pytest.skip("the library was not built")
    root = tmp_path / "tree"
    (root / "llvq_amd").mkdir(parents=True)
    (root / "llvq_amd" / "_calls.so").write_bytes(b"older")
    made = []

    def make(cmd):
        made.append(cmd)
        if "../_calls.so" in cmd:
            raise subprocess.CalledProcessError(2, cmd)

    monkeypatch.setattr(entry, "_ROOT", str(root))
    monkeypatch.setattr(entry.subprocess, "check_call", make)
    entry.build()
    assert any("liboracle.so" in c for c in made) and not (root / "llvq_amd" / "_calls.so").exists()
    assert "was not built" in capsys.readouterr().err
    shutil.rmtree(root)
