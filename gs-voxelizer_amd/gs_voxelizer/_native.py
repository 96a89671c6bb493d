"""The native autograd nodes (csrc/autograd.cpp) and which calls may take them.

Plain calls of ``optim_to_render`` and ``voxelize_gaussians`` (ordinary tensors,
no transform or mode active) go to ``project`` and ``voxelize``, which return
nothing for a call they do not take; the Python autograd classes then do it, and
raise its errors.  Without a module built for this torch, or in a torch that no
longer has one of the private names that `plain` asks, the classes do all calls
(same kernels and results, more host time), after a warning.
"""
import ctypes
import warnings

import torch
from torch.autograd import forward_ad

from . import _lib

_ENTRIES = ("gsv_status_string", "gsv_last_hip_error", "gsv_project_fwd", "gsv_project_bwd",
            "gsv_cumsum_bin_workspace_bytes", "gsv_cumsum_bin_and_sort_device_count",
            "gsv_voxelize_fwd", "gsv_voxelize_fwd_l1_workspace_bytes", "gsv_voxelize_fwd_l1",
            "gsv_voxelize_bwd_workspace_bytes", "gsv_voxelize_bwd", "gsv_voxelize_bwd_l1")

_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _load():
    """(module, None), or (None, why there is none)."""
    try:
        from . import _autograd
    except ImportError as e:  # not built, or against another torch's symbols
        return None, str(e)
    built_for = getattr(_autograd, "torch_version", None)
    if built_for is None:
        return None, "_autograd.so is of an older build"
    if built_for != torch.__version__:
        return None, f"built for torch {built_for}, this is {torch.__version__}"
    try:
        torch.compiler.is_compiling, torch._C._are_functorch_transforms_active
        torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack
        forward_ad._current_level, torch._C._get_tracing_state
    except AttributeError as e:
        return None, str(e)
    L = _lib.load()
    _autograd.bind({name: ctypes.cast(getattr(L, name), ctypes.c_void_p).value
                    for name in _ENTRIES})
    return _autograd, None


_module, _why = _load()
available = _module is not None
if available:
    project, voxelize = _module.project, _module.voxelize
else:
    warnings.warn(f"gs_voxelizer: no native autograd nodes ({_why}); every call takes the Python "
                  "classes. Build them with `python gs-voxelizer_amd/build.py`.", RuntimeWarning)


def plain(*tensors) -> bool:
    """Whether there are native nodes, every argument is an ordinary tensor and
    nothing watches or transforms the call: no subclass, torch.func transform,
    forward-mode level, trace, compilation, or dispatch or function mode.
    (Saved-tensor hooks and anomaly mode act on native nodes as on Python ones.)"""
    if not available:
        return False
    for t in tensors:
        if type(t) not in _PLAIN:
            return False
    return not (torch.compiler.is_compiling() or torch._C._are_functorch_transforms_active()
                or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()
                or forward_ad._current_level >= 0 or torch._C._get_tracing_state() is not None)
