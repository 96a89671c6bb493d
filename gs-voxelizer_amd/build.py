"""Build libgsvox.so (gfx950) and the native autograd nodes in-tree:
``python gs-voxelizer_amd/build.py``.

hipcc compiles every ``csrc/*.hip`` for ``--offload-arch=gfx950`` and links one
C-ABI shared library next to the Python package, where ``gs_voxelizer._lib``
loads it.  No torch headers are involved, so the library is independent of the
torch build's C++ ABI.  csrc/autograd.cpp (host code, g++) is the part that does
use them: a Python extension module, gs_voxelizer/_autograd.so.  Where it cannot
be built (no torch headers, no g++) the library is built all the same, and
gs_voxelizer runs its Python autograd classes.
"""
import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "gs_voxelizer", "libgsvox.so")
AUTOGRAD = os.path.join(HERE, "gs_voxelizer", "_autograd.so")
SOURCES = ["scan.hip", "project.hip", "binning.hip", "voxelize.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # keep the compiler from forming packed-FP32 VALU instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]

# Per-source additions.  voxelize.hip runs in binary32 flush-to-zero mode: its
# forward builds exp2 values as products and relies on v_mul_f32 returning 0
# below 2^-126, the same gate v_exp_f32 applies (project.hip keeps IEEE
# denormals: its tile boxes are bit-exact with the reference).
SOURCE_FLAGS = {
    "voxelize.hip": ["-fgpu-flush-denormals-to-zero"],
}


def hipcc():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found; the gfx950 library cannot be built")


def _clean(text):
    # hipcc's host pass does not know the device-only target feature; drop that noise
    noise = ("unknown target feature", "packed-fp32-ops")
    return "\n".join(l for l in text.splitlines() if not any(k in l for k in noise))


def autograd_command(out):
    """The g++ command of the native autograd nodes against the installed torch."""
    import torch
    base = os.path.dirname(torch.__file__)
    include = [os.path.join(base, "include"),
               os.path.join(base, "include", "torch", "csrc", "api", "include"),
               os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"),
               sysconfig.get_paths()["include"]]
    return ([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
             "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_EXTENSION_NAME=_autograd",
             f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
             f'-DGSV_TORCH_VERSION="{torch.__version__}"']
            + ["-isystem" + d for d in include]
            + [os.path.join(CSRC, "autograd.cpp"), "-o", out, "-L" + os.path.join(base, "lib"),
               "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python"])


def _start_autograd(out, verbose):
    """The running g++ of the autograd module, or the reason why there is none."""
    try:
        cmd = autograd_command(out)
        if verbose:
            print(" ".join(cmd), flush=True)
        return subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    except (ImportError, AttributeError, OSError) as e:
        return f"{type(e).__name__}: {e}"


def _install_autograd(started, out, verbose):
    """Puts the autograd module in place; without one an older module goes too."""
    if not isinstance(started, str):
        log = started.communicate()[0]
        if started.returncode == 0:
            if verbose and log.strip():
                print(log, flush=True)
            os.replace(out, AUTOGRAD)
            return
        started = f"g++ ({started.returncode}):\n{log}"
    if os.path.exists(AUTOGRAD):
        os.remove(AUTOGRAD)
    print(f"the native autograd nodes were not built: {started}", file=sys.stderr, flush=True)


def build(verbose=False):
    """Compile the library and the autograd module; returns the library's path.
    Always recompiles.  Raises where the library cannot be built; without the
    autograd module it says why on stderr.

    Each source is compiled to an object in its own hipcc process (they run
    concurrently; every translation unit is self-contained), then one link
    step writes the shared library.
    """
    flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    with tempfile.TemporaryDirectory(dir=os.path.dirname(OUT)) as tmpdir:
        procs, tmp_autograd = [], os.path.join(tmpdir, "_autograd.so")
        autograd = _start_autograd(tmp_autograd, verbose)
        for s in SOURCES:
            obj = os.path.join(tmpdir, os.path.splitext(s)[0] + ".o")
            cmd = [hipcc()] + flags + SOURCE_FLAGS.get(s, []) + ["-c", os.path.join(CSRC, s), "-o", obj]
            if verbose:
                print(" ".join(cmd), flush=True)
            procs.append((s, obj, subprocess.Popen(cmd, stdout=subprocess.PIPE,
                                                   stderr=subprocess.STDOUT, text=True)))
        failed, objs = [], []
        for s, obj, pr in procs:
            out, _ = pr.communicate()
            log = _clean(out)
            if pr.returncode != 0:
                failed.append(f"{s} ({pr.returncode}):\n{log}")
            elif verbose and log.strip():
                print(log, flush=True)
            objs.append(obj)
        if failed:
            if not isinstance(autograd, str):
                autograd.communicate()
            raise RuntimeError("hipcc failed: " + "\n".join(failed))
        tmp = os.path.join(tmpdir, "libgsvox.so")
        cmd = [hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", tmp]
        if verbose:
            print(" ".join(cmd), flush=True)
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError(f"hipcc link failed ({res.returncode}):\n{_clean(res.stdout + res.stderr)}")
        os.replace(tmp, OUT)
        _install_autograd(autograd, tmp_autograd, verbose)
    return OUT


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
