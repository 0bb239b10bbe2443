"""Builds libmamba_ss.so, the HIP selective-scan library, for gfx950, and
mamba_host.so, the native host side of the Python layer.

``python -m mamba_amd.build`` (or ``build()``) compiles every source under
``mamba_amd/csrc`` with hipcc (one object per source, in parallel) and links
them into ``mamba_amd/_lib/libmamba_ss.so``.  The library is built in-tree
so that it travels with the source tree.
"""
import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "_lib")
OBJ_DIR = os.path.join(LIB_DIR, "obj")
LIB_PATH = os.path.join(LIB_DIR, "libmamba_ss.so")
HOST_PATH = os.path.join(LIB_DIR, "mamba_host.so")
ARCH = os.environ.get("MAMBA_AMD_ARCH", "gfx950")
# the scan kernels are one unit per I/O type (the units without a suffix hold fp32's)
SOURCES = ["ss_bwd.hip", "ss_bwd_bf16.hip", "ss_bwd_f16.hip", "ss_fwd.hip", "ss_fwd_bf16.hip", "ss_fwd_f16.hip",
           "ss_api.hip", "conv1d.hip", "rms_norm.hip", "decode.hip", "decode_linear.hip"]


def hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or install ROCm)")


def compile_flags():
    return [
        f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
        # packed fp32 VALU ops are disabled on purpose: the scan is written in
        # scalar fp32 and must not be vectorised into v_pk_* forms
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        "-Wall", "-Wno-unused-function",
        "-I", os.path.join(HERE, "..", "include"),
    ]


def host_cxx():
    for cand in (os.environ.get("CXX"), shutil.which("g++"), shutil.which("c++")):
        if cand and shutil.which(cand):
            return cand
    raise RuntimeError("no host C++ compiler found (set CXX)")


def torch_dir(name):
    import torch
    return os.path.join(os.path.dirname(torch.__file__), name)


def host_flags():
    """Flags of the host module (csrc/host_ops.cpp), a torch C++ extension without device code."""
    import torch
    inc = torch_dir("include")
    return ["-O2", "-std=c++17", "-fPIC", "-Wall", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            "-I", inc, "-I", os.path.join(inc, "torch", "csrc", "api", "include"),
            "-I", sysconfig.get_paths()["include"], "-I", os.path.join(HERE, "..", "include")]


def build_command(out=LIB_PATH):
    """One hipcc command that compiles and links everything (for reference)."""
    return [hipcc()] + compile_flags() + ["-shared", "-o", out] + [os.path.join(CSRC, s) for s in SOURCES]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{' '.join(cmd)}\n{res.stderr[-8000:]}")


def build(verbose=False, jobs=None):
    os.makedirs(OBJ_DIR, exist_ok=True)
    cc = hipcc()
    objs = [os.path.join(OBJ_DIR, os.path.splitext(s)[0] + ".o") for s in SOURCES]
    cmds = [[cc] + compile_flags() + ["-c", "-o", o, os.path.join(CSRC, s)] for s, o in zip(SOURCES, objs)]
    # the host module's one unit beside them (g++: host code only)
    host_obj = os.path.join(OBJ_DIR, "host_ops.o")
    pool = ThreadPoolExecutor(max_workers=1)
    host = pool.submit(_run, [host_cxx()] + host_flags() + ["-c", "-o", host_obj, os.path.join(CSRC, "host_ops.cpp")],
                       verbose)
    jobs = jobs or min(len(cmds), max(1, min(16, os.cpu_count() or 1)))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        list(ex.map(lambda c: _run(c, verbose), cmds))
    tmp = LIB_PATH + ".tmp"
    _run([cc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs, verbose)
    os.replace(tmp, LIB_PATH)
    host.result()
    pool.shutdown()
    tmp = HOST_PATH + ".tmp"
    _run([host_cxx(), "-shared", "-o", tmp, host_obj, "-L", torch_dir("lib"), "-ltorch_python", "-ltorch", "-ltorch_cpu",
          "-lc10", "-L", LIB_DIR, "-lmamba_ss", "-Wl,-rpath,$ORIGIN"], verbose)
    os.replace(tmp, HOST_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
