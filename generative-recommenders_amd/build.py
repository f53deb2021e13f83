"""Compile ``csrc/`` into ``csrc/libhstu_hip.so`` and ``csrc/libhstu_linear.so`` with hipcc for gfx950 (cross-compiles
without a GPU), and ``csrc/hstu_native.so``, the operators' native front, with the host compiler."""

import os
import shutil
import subprocess
import sysconfig

_HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(_HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(_HERE), "include")
LIB_PATH = os.path.join(CSRC, "libhstu_hip.so")
LINEAR_LIB_PATH = os.path.join(CSRC, "libhstu_linear.so")  # separate: it links hipBLASLt, the attention library does not
NATIVE_PATH = os.path.join(CSRC, "hstu_native.so")  # links the two above and libtorch; finds them beside itself

# -packed-fp32-ops off: hipcc must not fuse scalar float code into v_pk_*_f32 on this hardware pool.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-fPIC",
    "-shared",
]


def _run(cmd, verbose):
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + " ".join(cmd) + "\n" + proc.stdout + proc.stderr)
    if verbose:
        print(" ".join(cmd))


def _native_commands():
    """Compile and link commands of the native front (host code only: the linking needs the two libraries)."""
    import torch

    root = os.path.dirname(torch.__file__)
    obj = os.path.join(CSRC, "hstu_native.o")
    cxx = shutil.which("g++") or "c++"
    includes = [f"-I{INCLUDE}"]
    for path in (os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"), "/opt/rocm/include",
                 sysconfig.get_paths()["include"]):
        includes += ["-isystem", path]
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    compile_ = [cxx, "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-DTORCH_API_INCLUDE_EXTENSION_H",
                "-DTORCH_EXTENSION_NAME=hstu_native", f"-D_GLIBCXX_USE_CXX11_ABI={abi}", *includes, "-c", os.path.join(CSRC, "hstu_native.cpp"), "-o", obj]
    link = [cxx, "-shared", obj, "-o", NATIVE_PATH, f"-L{CSRC}", "-l:libhstu_hip.so", "-l:libhstu_linear.so", "-L" + os.path.join(root, "lib"),
            "-lc10", "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]
    return compile_, link, obj


def build_library(verbose: bool = False) -> str:
    """Always recompiles; returns the path of the attention library.  The translation units compile side by side
    (attention forward and backward, dense steps forward and backward, native front), then the two libraries are linked
    and the front against both."""
    from concurrent.futures import ThreadPoolExecutor

    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    common = [hipcc] + [f for f in HIPCC_FLAGS if f != "-shared"] + ["-I", INCLUDE, "-I", CSRC]
    objs = [os.path.join(CSRC, name) for name in ("hstu_api.o", "hstu_bwd_api.o", "hstu_fwd_fitted.o", "hstu_bwd_f32.o")]
    linear_objs = [os.path.join(CSRC, "hstu_linear.o"), os.path.join(CSRC, "hstu_linear_bwd.o"), os.path.join(CSRC, "hstu_uqvk.o"),
                   os.path.join(CSRC, "hstu_uqvk_bwd.o")]
    jobs = [
        common + ["-c", os.path.join(CSRC, "hstu_api.hip"), "-o", objs[0]],
        common + ["-c", os.path.join(CSRC, "hstu_bwd_api.hip"), "-o", objs[1]],
        common + ["-c", os.path.join(CSRC, "hstu_fwd_fitted.hip"), "-o", objs[2]],
        common + ["-c", os.path.join(CSRC, "hstu_bwd_f32.hip"), "-o", objs[3]],
        common + ["-c", os.path.join(CSRC, "hstu_linear.hip"), "-o", linear_objs[0]],
        common + ["-c", os.path.join(CSRC, "hstu_linear_bwd.hip"), "-o", linear_objs[1]],
        # (matrix results in vector registers: see the file)
        common + ["-mllvm", "-amdgpu-mfma-vgpr-form", "-c", os.path.join(CSRC, "hstu_uqvk.hip"), "-o", linear_objs[2]],
        common + ["-mllvm", "-amdgpu-mfma-vgpr-form", "-c", os.path.join(CSRC, "hstu_uqvk_bwd.hip"), "-o", linear_objs[3]],
    ]
    native_compile, native_link, native_obj = _native_commands()
    jobs.append(native_compile)
    with ThreadPoolExecutor(max_workers=8) as pool:
        list(pool.map(lambda c: _run(c, verbose), jobs))
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", LIB_PATH], verbose)
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + linear_objs + ["-o", LINEAR_LIB_PATH, "-lhipblaslt"], verbose)
    _run(native_link, verbose)
    for o in objs + linear_objs + [native_obj]:
        os.remove(o)
    return LIB_PATH
