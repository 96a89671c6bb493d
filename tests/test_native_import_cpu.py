"""The native autograd nodes are an addition to the Python classes: the package
imports without them, with a module of another torch or of an older build, or in a
torch without one of the private names that decide which calls are plain, and says
so once."""
import os
import subprocess
import sys

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gs-voxelizer_amd")

MISSING = """
import sys
sys.modules["gs_voxelizer._autograd"] = None  # import raises ModuleNotFoundError
"""
OTHER_TORCH = """
import sys, types
m = types.ModuleType("gs_voxelizer._autograd")
m.torch_version = "1.0.0"
sys.modules["gs_voxelizer._autograd"] = m
"""
OLDER_BUILD = """
import sys, types
sys.modules["gs_voxelizer._autograd"] = types.ModuleType("gs_voxelizer._autograd")
"""


def _without(owner, name):
    return (f"import torch, torch.autograd.forward_ad\nsaved = {owner}.{name}\n"
            f"delattr({owner}, {name!r})\n"
            f"restore = lambda: setattr({owner}, {name!r}, saved)  # torch itself uses some\n", name)


@pytest.mark.parametrize("before,why", [
    (MISSING, "_autograd"), (OTHER_TORCH, "torch 1.0.0"), (OLDER_BUILD, "an older build"),
    _without("torch._C", "_are_functorch_transforms_active"),
    _without("torch._C", "_len_torch_dispatch_stack"),
    _without("torch._C", "_len_torch_function_stack"),
    _without("torch._C", "_get_tracing_state"),
    _without("torch.autograd.forward_ad", "_current_level"),
    _without("torch.compiler", "is_compiling")],
    ids=["missing", "other_torch", "older_build", "transforms", "dispatch", "function", "trace",
         "forward_mode", "compile"])
def test_the_package_imports_without_the_nodes(before, why):
    code = before + """
import torch
import gs_voxelizer.optim_to_render as o, gs_voxelizer.voxelize, gs_voxelizer.graph
from gs_voxelizer import _native
if "restore" in globals():
    restore()
assert not _native.available and not _native.plain(torch.zeros(1))
z = torch.zeros((0, 3))
try:
    o.optim_to_render(z, z, torch.zeros((0, 4)), torch.zeros((0, 1)), (8, 8, 8), (1.0, 1.0, 1.0),
                      (0.5, 0.5, 0.5))
except ValueError as e:
    print(e)
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                       env=dict(os.environ, PYTHONPATH=PKG))
    assert r.returncode == 0, r.stderr
    assert "Invalid shape" in r.stdout
    assert r.stderr.count("RuntimeWarning: gs_voxelizer: no native") == 1 and why in r.stderr
