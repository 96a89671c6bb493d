"""The package installs with pip the way the reference's does (setup.py:153-179
of PaPieta/gs-voxelizer): metadata, the package list and the compiled library
as package data.  Reading the metadata does not compile anything."""
import importlib.util
import os
import shutil
import subprocess
import sys

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gs-voxelizer_amd")


def test_setup_metadata_lists_the_library():
    out = subprocess.run([sys.executable, "setup.py", "--name", "--version"], cwd=PKG,
                         capture_output=True, text=True, check=True).stdout.split()
    assert out[-2:] == ["gs-voxelizer-amd", "0.2.0"]
    import gs_voxelizer
    assert gs_voxelizer.__version__ == "0.2.0"
    with open(os.path.join(PKG, "setup.py")) as f:
        text = f.read()
    assert '"libgsvox.so"' in text and "build_py" in text
    assert os.path.exists(os.path.join(PKG, "pyproject.toml"))


def _raise_import_error(out):
    raise ImportError("no torch")


@pytest.mark.skipif(not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")),
                    reason="hipcc not installed")
@pytest.mark.parametrize("command", [_raise_import_error, lambda out: ["false"],
                                     lambda out: ["no-such-compiler"]])
def test_the_library_is_built_without_the_autograd_module(tmp_path, monkeypatch, capfd, command):
    """The C-ABI library needs neither torch nor g++: a box without them gets it,
    a line on stderr, and no module of an earlier build."""
    spec = importlib.util.spec_from_file_location("gsv_build", os.path.join(PKG, "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    out, stale = tmp_path / "libgsvox.so", tmp_path / "_autograd.so"
    stale.write_text("older")
    monkeypatch.setattr(mod, "OUT", str(out))
    monkeypatch.setattr(mod, "AUTOGRAD", str(stale))
    monkeypatch.setattr(mod, "SOURCES", ["scan.hip"])
    monkeypatch.setattr(mod, "autograd_command", command)
    assert mod.build() == str(out)
    assert out.exists() and not stale.exists()
    assert "autograd nodes were not built" in capfd.readouterr().err
