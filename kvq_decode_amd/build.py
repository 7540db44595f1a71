"""Build libkvq.so (the HIP kernels + C ABI) in-tree for gfx950, and _host.so, the native
host path of the Python entry points.

    python -m kvq_decode_amd.build          # or: python kvq_decode_amd/build.py

Compiles csrc/*.hip and csrc/*.cpp with hipcc (one process per source, in parallel) and
links kvq_decode_amd/libkvq.so. Always recompiles (the build check runs it on every call);
a failed compile raises.
"""
import os
import shutil
import subprocess
import sys
import time
import warnings
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_DIR = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
INCLUDE = os.path.join(REPO_DIR, "include")
LIB_PATH = os.path.join(PKG_DIR, "libkvq.so")
HOST_PATH = os.path.join(PKG_DIR, "_host.so")
OBJ_DIR = os.path.join(PKG_DIR, "_build")  # objects (not committed, not shipped)

ARCH = "gfx950"
SOURCES = ["capi.cpp", "decode.hip", "decode_q.hip", "decode_q_d64.hip", "decode_q_d256.hip",
           "quant.hip", "append.hip", "static_workspace.hip"]

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # Packed fp32 VALU ops (v_pk_{add,mul,fma}_f32) stay off: hipcc would otherwise form
    # them from ordinary float code. The host pass warns that it does not know the feature.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA accumulators in VGPRs: the softmax rescale works on them with VALU ops, which
    # would otherwise copy them out of and back into AGPRs every chunk.
    "-mllvm", "-amdgpu-mfma-vgpr-form",
    # No -ffast-math: fp32 division stays correctly rounded (the quantizer's codes must be
    # bit-exact with its float32 spec; quant.hip also turns fp contraction off).
]


def hipcc():
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    return os.environ.get("HIPCC", os.path.join(rocm, "bin", "hipcc"))


def _compile(src, obj, cmd_base):
    cmd = [*cmd_base, "-c", src, "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    return proc, cmd


def host_needs():
    """What csrc/host.cpp needs and this machine lacks (None: nothing): a C++ compiler and the
    C++ headers of torch and Python, which hipcc and the kernels do without."""
    import sysconfig

    import torch
    cxx = os.environ.get("CXX", "g++")
    if shutil.which(cxx) is None:
        return f"the C++ compiler {cxx}"
    for path in (os.path.join(os.path.dirname(torch.__file__), "include", "ATen", "ATen.h"),
                 os.path.join(sysconfig.get_paths()["include"], "Python.h")):
        if not os.path.exists(path):
            return path
    return None


def host_command(out):
    """The compiler call for csrc/host.cpp: host code against torch's C++ headers."""
    import sysconfig

    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    lib = os.path.join(root, "lib")
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared",
            "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            f"-I{root}/include", f"-I{root}/include/torch/csrc/api/include", f"-I{rocm}/include",
            f"-I{sysconfig.get_paths()['include']}", f"-I{INCLUDE}",
            os.path.join(CSRC, "host.cpp"), "-o", out, f"-L{lib}", f"-Wl,-rpath,{lib}",
            "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python"]


def _filter(proc):
    noise = ("packed-fp32-ops", "is not a recognized feature")
    return [ln for ln in (proc.stdout + proc.stderr).splitlines()
            if not any(n in ln for n in noise)]


def build(verbose=False):
    """Compiles every source to an object in parallel (one hipcc per source), then links
    libkvq.so. The kernels of different sources call nothing across files, so no
    relocatable device code is needed. A machine that cannot compile the native host path
    builds libkvq.so alone, with a warning; a compile that fails raises."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    base = [hipcc(), *flags, f"-I{INCLUDE}", f"-I{CSRC}"]
    t0 = time.time()
    jobs = [(os.path.join(CSRC, s), os.path.join(OBJ_DIR, s + ".o")) for s in SOURCES]
    host_tmp = HOST_PATH + ".tmp"
    missing = host_needs()
    with ThreadPoolExecutor(max_workers=min(len(jobs) + 1, os.cpu_count() or 1)) as pool:
        if missing is None:
            host_cmd = host_command(host_tmp)
            host = pool.submit(subprocess.run, host_cmd, capture_output=True, text=True)
        results = list(pool.map(lambda j: _compile(j[0], j[1], base), jobs))
        if missing is None:
            results.append((host.result(), host_cmd))
    msgs = []
    for proc, cmd in results:
        msgs += _filter(proc)
        if proc.returncode != 0:
            raise RuntimeError("compiler failed (%d):\n%s\ncommand: %s"
                               % (proc.returncode, "\n".join(_filter(proc)), " ".join(cmd)))
    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC",
           *[o for _, o in jobs], "-o", tmp]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError("link failed (%d):\n%s\ncommand: %s"
                           % (proc.returncode, "\n".join(_filter(proc)), " ".join(cmd)))
    os.replace(tmp, LIB_PATH)
    if missing is None:
        os.replace(host_tmp, HOST_PATH)
    else:
        if os.path.exists(HOST_PATH):  # built from other sources than libkvq.so
            os.remove(HOST_PATH)
        warnings.warn(f"{HOST_PATH} was not built ({missing} not found): the Python entry points "
                      "work without it, at more host time per call", RuntimeWarning)
    if verbose:
        for m in msgs:
            print(m)
        print(f"built {LIB_PATH} in {time.time() - t0:.1f}s")
    build_checks(verbose)
    return LIB_PATH


# GPU check programs of the test suite (tests/gpu_checks/*.hip -> executables beside them)
CHECKS_DIR = os.path.join(REPO_DIR, "tests", "gpu_checks")


def build_checks(verbose=False):
    if not os.path.isdir(CHECKS_DIR):
        return
    for name in sorted(os.listdir(CHECKS_DIR)):
        if not name.endswith(".hip"):
            continue
        src = os.path.join(CHECKS_DIR, name)
        out = src[:-len(".hip")]
        cmd = [hipcc(), f"--offload-arch={ARCH}", "-O3", "-std=c++17",
               "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               f"-I{INCLUDE}", f"-I{CSRC}", src, "-o", out]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError("hipcc failed (%d) on %s:\n%s"
                               % (proc.returncode, src, proc.stderr[-3000:]))
        if verbose:
            print(f"built {out}")


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
