"""Builds libw8a8.so (every HIP source under csrc/) for gfx950 with hipcc, and, where g++ and a ROCm torch
with its headers are there, the _launch module (the wrappers' launch path, csrc/bind.cpp).

Run as `python -m w8a8.build` from gemma-npu_amd/, or through __graft_entry__.build().
Objects go to gemma-npu_amd/_build/, the library next to this file.
"""
import concurrent.futures
import glob
import os
import shutil
import subprocess
import sys
import sysconfig

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(ROOT, "csrc")
INCLUDE = os.path.join(os.path.dirname(ROOT), "include")
BUILD = os.path.join(ROOT, "_build")
LIB = os.path.join(PKG, "libw8a8.so")
LAUNCH = os.path.join(PKG, "_launch" + sysconfig.get_config_var("EXT_SUFFIX"))
ARCH = "gfx950"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17", "-Wall", "-Wno-unused-function",
    # Evaluate a * b + c as the two roundings the reference performs, never as one fused op.
    "-ffp-contract=off",
    # Keep hipcc from forming packed fp32 (v_pk_*_f32) instructions.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{CSRC}",
    f"-I{INCLUDE}",
]


def _compile(src):
    obj = os.path.join(BUILD, os.path.basename(src) + ".o")
    cmd = [HIPCC, *CFLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def _build_launch():
    """csrc/bind.cpp (host code against torch's headers) -> LAUNCH, linked to libw8a8.so.  Returns None, or why
    it was left out: the wrappers then make every call through ctypes."""
    try:
        import torch
        from torch.utils import cpp_extension

        from w8a8 import _lib
    except ImportError as e:
        return f"{e}"
    if not torch.version.hip:
        return "torch is not built for ROCm"
    if not shutil.which("g++"):
        return "no g++"
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    include = [*cpp_extension.include_paths(), os.path.join(rocm, "include"), sysconfig.get_paths()["include"], INCLUDE]
    tmp = LAUNCH + ".tmp"
    fits = {"W8A8_TORCH": _lib.torch_build(), "W8A8_SOURCES": _lib.launch_sources()}
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           *(f'-D{k}="{v}"' for k, v in fits.items()),
           *(f"-isystem{d}" for d in include), os.path.join(CSRC, "bind.cpp"), "-o", tmp,
           f"-L{os.path.join(os.path.dirname(torch.__file__), 'lib')}", "-ltorch_python", "-ltorch", "-ltorch_cpu",
           "-ltorch_hip", "-lc10", "-lc10_hip", f"-L{os.path.join(rocm, 'lib')}", "-lamdhip64", f"-L{PKG}", "-lw8a8",
           "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        return f"g++ failed on bind.cpp:\n{r.stdout}\n{r.stderr}"
    os.replace(tmp, LAUNCH)
    return None


def build(verbose=False):
    os.makedirs(BUILD, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    # no launch path of another build beside the new library, whatever becomes of this one's
    for old in glob.glob(os.path.join(PKG, "_launch*.so")):
        os.remove(old)
    os.replace(tmp, LIB)
    left_out = _build_launch()
    if left_out:
        print(f"{LAUNCH} left out, the wrappers call through ctypes: {left_out}", flush=True)
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources" + ("" if left_out else f" and {LAUNCH}"), flush=True)
    return LIB


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    build(verbose=True)
    sys.exit(0)
