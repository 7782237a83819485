"""The host module (csrc/ktx_host.cpp) has torch's and the interpreter's layouts compiled in, and the package runs without it."""
import os
import sysconfig

import pytest
import torch

from ktransformers_amd import _native as n
from ktransformers_amd import build as b


def test_another_torch_or_interpreter_has_another_module(monkeypatch):
    here = b.host_lib()
    assert here.endswith(sysconfig.get_config_var("EXT_SUFFIX")) and torch.__version__ in os.path.basename(here)
    monkeypatch.setattr(torch, "__version__", "0.0.0")
    assert b.host_lib() != here and n._load_host() is None


def test_a_module_that_does_not_load_leaves_the_calls_to_python(monkeypatch, tmp_path):
    path = tmp_path / "ktx_host.so"
    path.write_bytes(b"no library")
    monkeypatch.setattr(b, "host_lib", lambda: str(path))
    with pytest.warns(RuntimeWarning, match="does not load"):
        assert n._load_host() is None


def test_the_library_is_built_where_the_module_cannot_be(monkeypatch, tmp_path, capsys):
    monkeypatch.setattr(b, "host_lib", lambda: str(tmp_path / "ktx_host.so"))
    monkeypatch.setattr(b, "_build_lib", lambda force, verbose: b.LIB)
    for compiler in ("false", "/no/such/compiler"):
        monkeypatch.setenv("CXX", compiler)
        assert b.build() == b.LIB and not (tmp_path / "ktx_host.so").exists()
        assert "was not built" in capsys.readouterr().err
