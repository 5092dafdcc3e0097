"""What the build leaves when torch does not let _calls.so be built: the C library needs no torch."""
import importlib.util
import subprocess

import pytest


@pytest.mark.parametrize("torch_there", [True, False])
def test_the_library_is_linked_without_the_calls(monkeypatch, tmp_path, torch_there):
    from candle_amd import build
    linked = []
    monkeypatch.setattr(build, "LIB_DIR", str(tmp_path))
    monkeypatch.setattr(build, "_compile", lambda src: src)
    find = importlib.util.find_spec
    monkeypatch.setattr(importlib.util, "find_spec", lambda name, *a: None if name == "torch" and not torch_there else find(name, *a))

    def run(cmd, **kw):
        if build.CALLS_PATH in cmd:
            raise subprocess.CalledProcessError(1, cmd)   # a torch without what the source includes
        linked.append(cmd[cmd.index("-o") + 1])
    monkeypatch.setattr(subprocess, "check_call", run)
    if torch_there:
        with pytest.raises(subprocess.CalledProcessError):   # a build that failed says so, with the libraries in place
            build.build(verbose=False)
    else:
        assert build.build(verbose=False) == build.LIB_PATH   # nobody can load the module there
    assert linked == [build.LIB_PATH, build.PROBE_LIB_PATH]
