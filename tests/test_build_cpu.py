"""llmmm_amd/build.py without compilers: what it builds when the Python side cannot be built."""
import importlib.util
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_c_library_is_linked_without_torch(monkeypatch, tmp_path):
    """A user of include/llmmm.h on a machine without torch or g++: the build says what is missing, and libllmmm.so is there."""
    spec = importlib.util.spec_from_file_location("_llmmm_build", os.path.join(ROOT, "llmmm_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    linked = []

    def no_binding():
        raise ImportError("No module named 'torch'")

    def run(cmd, **kw):
        linked.append((cmd[0], cmd[cmd.index("-o") + 1]))
        return subprocess.CompletedProcess(cmd, 0, stdout="")

    monkeypatch.setattr(build, "OBJ", str(tmp_path))
    monkeypatch.setattr(build, "_compile", lambda item: (str(tmp_path / item[0]), ""))
    monkeypatch.setattr(build, "_compile_binding", no_binding)
    monkeypatch.setattr(build.subprocess, "run", run)
    with pytest.raises(ImportError, match="torch"):
        build.build()
    assert linked == [("hipcc", build.LIB)]
