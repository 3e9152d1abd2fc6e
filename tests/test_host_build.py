"""The native host module's build and load (csrc/Makefile, _lib.host): named after the torch and the interpreter it is for, never what stops the build, and missed aloud."""
import os
import subprocess
import sys
import sysconfig
import types

import pytest
import torch

from gbx_lm_amd import _lib

CSRC = os.path.dirname(_lib.host_so_path())


def _make(*args):
    return subprocess.run(["make", "-C", CSRC, *args], capture_output=True, text=True, timeout=120)


def test_the_name_holds_torch_and_the_interpreter():
    name = os.path.basename(_lib.host_so_path())
    assert torch.__version__ in name and name.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
    shown = _make("-n", "-B", "host", f"PY={sys.executable}")
    assert shown.returncode == 0 and f"mv -f {name}.tmp {name}" in shown.stdout


def test_an_interpreter_without_torch_does_not_stop_the_build():
    done = _make("host", "PY=false")
    assert done.returncode == 0 and "not built" in done.stderr


def test_a_compile_that_fails_does_not_stop_the_build(tmp_path):
    target = tmp_path / "host.so"
    target.write_bytes(b"of an older source")
    os.utime(target, (0, 0))
    done = _make("host", f"PY={sys.executable}", "CXX=false", f"HLIB={target}")
    assert done.returncode == 0 and "not built" in done.stderr
    assert os.listdir(tmp_path) == []                                   # nor is the older source's module left to be loaded


@pytest.mark.parametrize("there", [False, True])
def test_a_module_that_is_missing_or_does_not_load_is_missed_aloud(tmp_path, monkeypatch, there):
    path = tmp_path / os.path.basename(_lib.host_so_path())
    if there:
        path.write_bytes(b"no shared object")
    monkeypatch.setattr(_lib, "host_so_path", lambda: str(path))
    monkeypatch.setattr(_lib, "lib", lambda: types.SimpleNamespace())
    monkeypatch.setattr(_lib, "_host", None)
    with pytest.warns(RuntimeWarning, match="does not load" if there else "is not built"):
        assert _lib.host() is None
    assert _lib.host() is None                                          # (once)
