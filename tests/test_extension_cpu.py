"""The optional extension of the Python mirror: building and loading the library do without it, and say so."""
import os
import subprocess
import sys
import warnings

import pytest

import lc0_amd
from lc0_amd import backend as be
from lc0_amd import build as lib_build


@pytest.mark.parametrize("error", [FileNotFoundError("g++"), subprocess.CalledProcessError(1, "g++")])
def test_without_a_compiler_or_headers_the_build_goes_on_and_no_old_extension_stays(error, tmp_path, monkeypatch, capfd):
    calls = tmp_path / "_calls.so"
    calls.write_bytes(b"of an earlier build")

    def fail(cmd, *args, **kwargs):
        raise error

    class Compiler:
        returncode = 0

        def __init__(self, cmd, **kwargs):
            pass

        def communicate(self):
            return "", None

    monkeypatch.setattr(lib_build, "CALLS", str(calls))
    monkeypatch.setattr(lib_build, "HERE", str(tmp_path))
    monkeypatch.setattr(lib_build.subprocess, "Popen", Compiler)
    monkeypatch.setattr(lib_build.subprocess, "check_call", lambda cmd: fail(cmd) if cmd[0] == "g++" else 0)
    assert lib_build.build() == lib_build.LIB
    assert not calls.exists()
    assert "_calls.so is not built" in capfd.readouterr().err


def test_an_extension_that_does_not_load_is_reported_and_an_absent_one_is_not(tmp_path, monkeypatch):
    monkeypatch.setitem(sys.modules, "lc0_amd._calls", None)   # (an import of it fails)
    monkeypatch.delattr(lc0_amd, "_calls", raising=False)
    monkeypatch.setattr(be, "_HERE", str(tmp_path))
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert be._load_calls() is None
    (tmp_path / os.path.basename(lib_build.CALLS)).write_bytes(b"")
    with pytest.warns(RuntimeWarning, match="does not load"):
        assert be._load_calls() is None
