"""Build libftnn_hip.so in-tree with hipcc for gfx950 (cross-compiles without a GPU), and the Python module over it."""
import importlib.machinery
import os
import shlex
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libftnn_hip.so")
SOURCES = ["ftnn_api.hip", "pack_kernels.hip", "mm_kernels.hip", "mfma_kernels.hip", "rows_kernels.hip", "stem_kernels.hip",
           "direct_kernels.hip", "ftnn_net.hip", "host_hash.cpp"]   # the last one is plain host C++
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wall", "-Wno-unused-function"]


# The tile GEMM kernels issue their LDS-direct loads through inline asm and count them by hand (s_waitcnt vmcnt(N)):
# every scratch access is itself a vector-memory operation that moves the count the waits rely on, so the build
# refuses scratch use in them (the library checks the same at run time before the first launch).  The layer kernels
# use ordinary loads that the compiler counts; scratch there would only be slow, and is refused as a performance guard.
# Source -> name fragments.
NO_SCRATCH = {"mfma_kernels.hip": ("k_conv_f4", "k_mfma"),   # "k_mfma" covers k_mfma_p4 as well
              "rows_kernels.hip": ("k_rows",), "direct_kernels.hip": ("k_direct_f4",)}


def check_no_scratch(src, remarks):
    """parse -Rpass-analysis=kernel-resource-usage remarks; raise if a listed kernel uses scratch"""
    name, bad, seen = None, [], {frag: 0 for frag in NO_SCRATCH[src]}
    for line in remarks.splitlines():
        if "remark: Function Name:" in line:
            name = line.split("Function Name:")[1].split()[0]
        elif "ScratchSize [bytes/lane]:" in line and name:
            for frag in NO_SCRATCH[src]:
                if frag in name:
                    seen[frag] += 1
                    if int(line.split("ScratchSize [bytes/lane]:")[1].split()[0]) != 0:
                        bad.append(name)
                    break
    missing = [frag for frag, n in seen.items() if n == 0]
    if bad or missing:
        raise RuntimeError("%s: %s" % (src, "kernels with scratch memory: %s" % bad if bad else
                                       "no resource remarks found for %s" % missing))


BINDING = os.path.join(HERE, "_call" + importlib.machinery.EXTENSION_SUFFIXES[0])


def binding_command():
    """the compiler call that makes _call from csrc/py_call.cpp (host code only), or what it needs that is not there"""
    try:
        import torch
    except ImportError as e:
        return None, str(e)
    root = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    cxx = shlex.split(os.environ.get("CXX", "g++"))
    include = sysconfig.get_paths()["include"]
    for what in (os.path.join(include, "Python.h"), os.path.join(root, "include", "c10", "hip", "HIPStream.h"), os.path.join(root, "lib", "libc10_hip.so")):
        if not os.path.exists(what):
            return None, "no " + what
    if not shutil.which(cxx[0]):
        return None, "no compiler " + cxx[0]
    inc = [include, os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"), os.path.join(rocm, "include")]
    return cxx + ["-O2", "-std=c++17", "-shared", "-fPIC", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                  "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI, '-DFTNN_TORCH="%s"' % torch.__version__] + ["-isystem" + d for d in inc] + [
        os.path.join(CSRC, "py_call.cpp"), "-o", BINDING, "-L" + HERE, "-lftnn_hip", "-Wl,-rpath,$ORIGIN", "-L" + os.path.join(root, "lib"),
        "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"], ""


def build_binding():
    """Compile the Python module; returns its path, or None where torch, Python's headers or a host compiler are missing (lib.py then
    makes every call through ctypes).  The library itself needs none of them."""
    cmd, missing = binding_command()
    if os.path.exists(BINDING):
        os.remove(BINDING)   # none is better than one of another library
    if cmd is None:
        print("%s is not built: %s" % (os.path.basename(BINDING), missing), file=sys.stderr)
        return None
    subprocess.run(cmd, check=True)
    return BINDING


def build_library(verbose=False):
    """Compile every HIP source and link the shared library, then the Python module where that can be; returns the library's path."""
    objs = []
    procs = []
    for src in SOURCES:
        obj = os.path.join(CSRC, os.path.splitext(src)[0] + ".o")
        objs.append(obj)
        cmd = [HIPCC] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
        if src.endswith(".cpp"):
            cmd = [HIPCC, "-x", "c++", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-c", os.path.join(CSRC, src), "-o", obj]
        if src in NO_SCRATCH:
            cmd.append("-Rpass-analysis=kernel-resource-usage")
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    for src, p in procs:
        out, _ = p.communicate()
        # the host pass does not know the packed-fp32 feature and says so; harmless
        out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l)
        if p.returncode != 0:
            raise RuntimeError("hipcc failed on %s:\n%s" % (src, out))
        if src in NO_SCRATCH:
            check_no_scratch(src, out)
            out = "\n".join(l for l in out.splitlines() if "kernel-resource-usage" not in l)
        if verbose and out.strip():
            print(out)
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", LIB]
    subprocess.run(cmd, check=True)
    build_binding()
    return LIB


if __name__ == "__main__":
    print(build_library(verbose="-v" in sys.argv))
