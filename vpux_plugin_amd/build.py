"""Builds libvpx_amd.so (HIP kernels + C ABI + host-side helpers) for gfx950, in-tree."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(HERE, "libvpx_amd.so")
BINDING = os.path.join(HERE, "_binding.so")

HIP_SOURCES = ["csrc/abi.hip", "csrc/sw_elementwise.hip", "csrc/sw_softmax.hip", "csrc/sw_mvn.hip", "csrc/sw_mvn_cminor.hip", "csrc/nce.hip", "csrc/nce_gemm.hip", "csrc/nce_gemm_regb.hip",
               "csrc/nce_direct.hip", "csrc/nce_conv_patch.hip", "csrc/nce_conv_rows.hip", "csrc/nce_conv_strips.hip", "csrc/nce_conv_regb.hip", "csrc/nce_conv_gather.hip", "csrc/nce_eltwise.hip", "csrc/calib.hip"]
HOST_SOURCES = ["host/compiler_utils.cpp"]

# -ffp-contract=off: fp32 expressions must round as written (FakeQuantize / Quantize parity).
# packed-fp32 VALU forms are switched off for every HIP translation unit.
HIP_FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-fvisibility=hidden",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wall", "-Wno-unused-function"]


def build(verbose=True, jobs=8):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    inc = ["-I", os.path.join(ROOT, "include"), "-I", os.path.join(HERE, "csrc")]
    procs = []
    objs = []
    for src in HIP_SOURCES + HOST_SOURCES:
        obj = os.path.join(objdir, os.path.basename(src) + ".o")
        objs.append(obj)
        cmd = [hipcc] + HIP_FLAGS + inc + ["-c", os.path.join(HERE, src), "-o", obj]
        if src.endswith(".cpp"):
            cmd = [hipcc, "-x", "hip"] + HIP_FLAGS + inc + ["-c", os.path.join(HERE, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
        if len(procs) >= jobs:
            _drain(procs, verbose)
    _drain(procs, verbose)
    # -no-hip-rt: no DT_NEEDED on a particular libamdhip64.  A process must hold exactly one HIP
    # runtime; the host application (or vpux_plugin_amd.runtime, which picks the copy torch ships)
    # provides it before this library is loaded.
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-no-hip-rt", "-o", LIB] + objs
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    # the C++ host example: the C ABI driven without Python; it links the HIP runtime itself
    exe = os.path.join(HERE, "examples", "c_abi_host")
    cmd = [hipcc, "--offload-arch=gfx950", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "examples", "c_abi_host.cpp"),
           "-L", HERE, "-lvpx_amd", "-Wl,-rpath,$ORIGIN/..", "-o", exe]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    build_binding(verbose)
    return LIB


def build_binding(verbose=True):
    """The CPython module runtime.py calls the library through: host code against torch's C++ headers.  torch's own
    libraries are in the process before it is loaded; libvpx_amd.so lies beside it.  A host that has only the C library to
    build lacks torch or the headers: it is told so, False is returned and the operator functions of runtime.py raise."""
    import sysconfig
    if os.path.exists(BINDING):
        os.remove(BINDING)  # (one of another build would call this library)
    python = sysconfig.get_paths()["include"]
    try:
        import torch
        top = os.path.dirname(torch.__file__)
        needs = [os.path.join(python, "Python.h"), os.path.join(top, "include", "torch", "csrc", "autograd", "python_variable.h")]
        absent = [h for h in needs if not os.path.exists(h)]
    except ImportError:
        absent = ["torch"]
    if absent:
        sys.stderr.write("%s is not built: %s not found (the C library and its hosts do not need it)\n" % (os.path.basename(BINDING), ", ".join(absent)))
        return False
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    # -DNDEBUG: torch's headers bring a counter of pybind11's with them otherwise, thread-local storage that no call comes to.  While a thread has not come
    # to the storage of the library that was loaded last, the C library (2.35) takes the long way for every lookup of every library in it: 0.1 ... 0.3 us a call.
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI, "-I", os.path.join(ROOT, "include")]
    for d in (os.path.join(top, "include"), os.path.join(rocm, "include"), python):
        cmd += ["-isystem", d]
    cmd += [os.path.join(HERE, "host", "torch_binding.cpp"), "-o", BINDING, "-L", HERE, "-lvpx_amd", "-Wl,-rpath,$ORIGIN",
            "-L", os.path.join(top, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return True


def _drain(procs, verbose):
    for src, p in procs:
        out, _ = p.communicate()
        text = out.decode(errors="replace")
        # the host pass does not know the device-only target feature; that warning is harmless
        text = "\n".join(l for l in text.splitlines() if "packed-fp32-ops" not in l and l.strip())
        if p.returncode != 0:
            sys.stderr.write(text + "\n")
            raise RuntimeError("compilation of %s failed" % src)
        if verbose and text:
            print(text, flush=True)
    procs.clear()


if __name__ == "__main__":
    build()
