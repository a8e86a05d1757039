"""Build liboptimus_mi355x.so (the C-ABI library) with hipcc for gfx950, and optimus_torch_host.so (the
C++ host module: allocations, launches and autograd nodes) with g++ against it.

    python optimus-lm_amd/build.py

Cross-compiles without a GPU.  The C-ABI library has no dependency on PyTorch: it exports plain
extern "C" functions over device pointers (see include/optimus_mi355x.h).
"""
import glob
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIBNAME = "liboptimus_mi355x.so"
HOSTNAME = "optimus_torch_host.so"

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # scalar fp32 arithmetic only: no packed-fp32 instruction selection
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def lib_path():
    return os.path.join(LIBDIR, LIBNAME)


def host_command(output):
    """g++ command for the host module's object file: host code only, PyTorch's headers."""
    import torch
    root = os.path.dirname(torch.__file__)
    include = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
               os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
    return ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DTORCH_EXTENSION_NAME=optimus_torch_host",
            *[f for d in include for f in ("-isystem", d)], "-c", os.path.join(CSRC, "host", "torch_host.cpp"), "-o", output]


def link_host(obj):
    import torch
    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    rocm = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib")
    out = os.path.join(LIBDIR, HOSTNAME)
    subprocess.run(["g++", "-shared", "-o", out, obj, "-L" + libs, "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu",
                    "-ltorch_python", "-L" + rocm, "-lamdhip64", "-L" + LIBDIR, "-l:" + LIBNAME, "-Wl,-rpath,$ORIGIN"],
                   check=True)
    return out


def build(verbose=False):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    os.makedirs(LIBDIR, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    objs = []
    procs = []
    objdir = os.path.join(LIBDIR, "obj")
    os.makedirs(objdir, exist_ok=True)
    compile_flags = [f for f in HIPCC_FLAGS if f != "-shared"]
    for s in srcs:
        o = os.path.join(objdir, os.path.basename(s)[:-4] + ".o")
        objs.append(o)
        cmd = [hipcc] + compile_flags + ["-c", s, "-o", o]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((s, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    host_obj = os.path.join(objdir, "torch_host.o")
    cmd = host_command(host_obj)
    if verbose:
        print(" ".join(cmd), flush=True)
    procs.append((cmd[-3], subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    failed = False
    for s, p in procs:
        out, _ = p.communicate()
        # hipcc's host pass does not know the device-only target feature; that warning is noise
        out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l and l.strip())
        if p.returncode != 0:
            failed = True
            print(f"[build] FAILED {s}\n{out}", file=sys.stderr)
        elif verbose and out:
            print(out)
    if failed:
        raise RuntimeError("a compiler failed")
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", lib_path()] + objs
    subprocess.run(cmd, check=True)
    link_host(host_obj)
    return lib_path()


if __name__ == "__main__":
    print(build(verbose=True))
