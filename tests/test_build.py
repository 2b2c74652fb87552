"""The build of the operator calls (kuiperllama_amd/build.py, build_pyops) beside the library's: without the interpreter's headers,
with sources that do not compile, for more than one interpreter."""
import os
import subprocess
import sysconfig

import pytest

from kuiperllama_amd import build, ops


@pytest.fixture
def elsewhere(tmp_path, monkeypatch):
    monkeypatch.setattr(build, "LIB_DIR", str(tmp_path))
    monkeypatch.setattr(build, "PYOPS_PATH", str(tmp_path / os.path.basename(build.PYOPS_PATH)))
    monkeypatch.setattr(ops, "_n", ops._n)  # a load binds it
    return tmp_path


def test_the_library_does_not_need_the_headers(elsewhere, monkeypatch, capsys):
    monkeypatch.setattr(sysconfig, "get_paths", lambda *a: {"include": str(elsewhere)})
    assert build.build_pyops(force=True) is None
    monkeypatch.setattr(build, "_stale", lambda: False)
    assert build.build_lib() == build.LIB_PATH
    assert capsys.readouterr().err.count("Python.h") == 2
    assert os.listdir(elsewhere) == []
    with pytest.raises(ImportError, match="headers"):
        ops._Unbound().add


def test_built_whole_under_the_interpreters_own_name(elsewhere, monkeypatch):
    path = build.build_pyops()
    assert path.endswith(sysconfig.get_config_var("EXT_SUFFIX")) and os.listdir(elsewhere) == [os.path.basename(path)]
    assert callable(ops._Unbound().add)
    before = open(path, "rb").read()
    bad = elsewhere / "csrc"
    bad.mkdir()
    (bad / "kh_pyops.c").write_text("#error no\n")
    monkeypatch.setattr(build, "CSRC", str(bad))
    with pytest.raises(subprocess.CalledProcessError):
        build.build_pyops(force=True)
    assert open(path, "rb").read() == before and sorted(os.listdir(elsewhere)) == ["csrc", os.path.basename(path)]
