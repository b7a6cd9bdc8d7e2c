"""Compile difflut_amd/csrc/*.hip into difflut_amd/lib/libdifflut_hip.so for gfx950 and csrc/host_ops.cpp, the autograd
functions over it, into difflut_amd/lib/difflut_host.so."""
import glob
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libdifflut_hip.so")
HOST_PATH = os.path.join(LIB_DIR, "difflut_host.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-munsafe-fp-atomics",  # float atomics as single hardware instructions
    # packed-fp32 instruction forms are kept out of every code object
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def sources():
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def host_command():
    """The compiler call for csrc/host_ops.cpp: host code against the installed torch."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    includes = cpp_extension.include_paths() + [sysconfig.get_paths()["include"], os.path.join(rocm, "include")]
    return (["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall", "-Wextra",
             "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
             "-D_GLIBCXX_USE_CXX11_ABI=" + str(int(torch._C._GLIBCXX_USE_CXX11_ABI)), "-DTORCH_API_INCLUDE_EXTENSION_H"]
            + [flag for d in includes for flag in ("-isystem", d)]  # (warnings of this source only, not of the headers)
            + [os.path.join(CSRC, "host_ops.cpp"), "-o", HOST_PATH, "-L" + torch_lib]
            + ["-l" + lib for lib in ("c10", "c10_hip", "torch_cpu", "torch_hip", "torch", "torch_python", "dl")]
            + ["-Wl,-rpath," + torch_lib])


def build(verbose=False, jobs=None):
    """Always recompiles (the sources in parallel, one compiler per file), then links; returns the path of the library."""
    from concurrent.futures import ThreadPoolExecutor

    os.makedirs(LIB_DIR, exist_ok=True)
    obj_dir = os.path.join(LIB_DIR, "_obj")
    os.makedirs(obj_dir, exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    compile_flags = [f for f in HIPCC_FLAGS if f != "-shared"] + ["-c"]

    def compile_one(src):
        obj = os.path.join(obj_dir, os.path.basename(src) + ".o")
        cmd = [hipcc] + compile_flags + ["-o", obj, src]
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError("hipcc failed on " + src + ":\n" + res.stdout + res.stderr)
        if verbose:
            print(" ".join(cmd))
        return obj

    def compile_host():
        cmd = host_command()
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError("g++ failed on host_ops.cpp:\n" + res.stdout + res.stderr)
        if res.stderr:
            print(res.stderr)
        if verbose:
            print(" ".join(cmd))

    srcs = sources()
    with ThreadPoolExecutor(max_workers=jobs or min(8, len(srcs) + 1)) as pool:
        host = pool.submit(compile_host)
        objs = list(pool.map(compile_one, srcs))
        host.result()
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH] + objs
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc (link) failed:\n" + res.stdout + res.stderr)
    if verbose:
        print(" ".join(cmd))
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
