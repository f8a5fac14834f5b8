"""Builds libdfa3d_hip.so for gfx950 with hipcc (cross-compiles without a GPU).

    python 3d-deformable-attention_amd/build.py [--force] [--clocks]

The library lands next to the python package (dfa3D/libdfa3d_hip.so) so that it travels with
the source tree, as does the module that calls it with torch's tensors (dfa3D/_binding.*.so, host code).  That module fits
one torch and one Python and is built again when either is another; where it cannot be built, calls go through ctypes.
Two more libraries land beside bench.py, which is what uses them: the yardstick kernels (libdfa3d_measure.so) and, with
--clocks, libdfa3d_hip_clocks.so: the same sources compiled with -DDFA3D_TILE_TIMING, i.e. with the per-phase clocks of the backward's tile kernels (`bench.py --phase-costs`).
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "dfa3D", "libdfa3d_hip.so")
BINDING_SRC = os.path.join(CSRC, "dfa3d_binding.cpp")
BINDING = os.path.join(HERE, "dfa3D", "_binding" + sysconfig.get_config_var("EXT_SUFFIX"))      # named for this Python
BINDING_STAMP = os.path.join(OBJ, "binding.built_for")
# yardstick kernels for bench.py (plain copy, bare gathers, LDS atomics, XCD map): not part of the operator library
MEASURE_SRC = os.path.join(CSRC, "measure", "dfa3d_measure.hip")
ROOT = os.path.dirname(HERE)
MEASURE_LIB = os.path.join(ROOT, "libdfa3d_measure.so")
CLOCKS_LIB = os.path.join(ROOT, "libdfa3d_hip_clocks.so")
CLOCKS_FLAGS = ["-DDFA3D_TILE_TIMING"]
SOURCES = ["dfa3d_forward.hip", "dfa3d_backward.hip", "dfa3d_backward_binned.hip", "dfa3d_backward_cells.hip",
           "dfa3d_rebatch.hip", "dfa3d_linear.hip", "dfa3d_locations.hip",
           "dfa3d_api.hip"]
HEADERS = ["dfa3d_device.h", "dfa3d_launch.h", "dfa3d_binned.h", os.path.join("..", "..", "include", "dfa3d.h")]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-munsafe-fp-atomics",
    # keep the compiler from forming packed fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def _stale(target, deps):
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)


def _build_lib(lib, obj_dir, extra_flags, force, verbose):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    os.makedirs(obj_dir, exist_ok=True)
    deps = [os.path.join(CSRC, h) for h in HEADERS] + [os.path.abspath(__file__)]
    jobs = []
    for src in SOURCES:
        s = os.path.join(CSRC, src)
        o = os.path.join(obj_dir, src.replace(".hip", ".o"))
        if force or _stale(o, deps + [s]):
            jobs.append([hipcc, *FLAGS, *extra_flags, "-c", s, "-o", o])
    with ThreadPoolExecutor(max_workers=5) as ex:
        list(ex.map(lambda cmd: _run(cmd, verbose), jobs))
    objs = [os.path.join(obj_dir, s.replace(".hip", ".o")) for s in SOURCES]
    if force or jobs or _stale(lib, objs):
        _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", lib, *objs], verbose)
    return lib


def _binding_stale(built_for):
    """`built_for`: the torch that is installed (dfa3D/_lib.py compares it with what the module was built for)."""
    if (_stale(BINDING, [BINDING_SRC, os.path.join(ROOT, "include", "dfa3d.h"), os.path.abspath(__file__)])
            or not os.path.exists(BINDING_STAMP)):
        return True
    with open(BINDING_STAMP) as f:
        return f.read() != built_for


def _build_binding(force, verbose):
    """Whether the module is there and up to date."""
    try:
        import torch
        from torch.utils import cpp_extension
        built_for = f"{torch.__version__} {torch.version.git_version}"
        if not (force or _binding_stale(built_for)):
            return True
        rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
        includes = [f"-isystem{d}" for d in [*cpp_extension.include_paths(), os.path.join(rocm, "include")]]
        libs = [f"-L{d}" for d in cpp_extension.library_paths()] + ["-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
        _run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall",
              f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f'-DDFA3D_BUILT_FOR="{built_for}"',
              "-I" + sysconfig.get_paths()["include"], *includes, BINDING_SRC, "-o", BINDING, *libs], verbose)
    except (ImportError, OSError, subprocess.CalledProcessError) as e:
        print(f"{BINDING} is not built ({e}): calls go through ctypes, which takes 5 to 10 us longer each", file=sys.stderr)
        if os.path.exists(BINDING):
            os.remove(BINDING)                   # of other sources or another torch
        return False
    os.makedirs(os.path.dirname(BINDING_STAMP), exist_ok=True)
    with open(BINDING_STAMP, "w") as f:
        f.write(built_for)
    return True


def build(force=False, verbose=True, clocks=False):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    with ThreadPoolExecutor(max_workers=1) as ex:
        binding = ex.submit(_build_binding, force, verbose)
        _build_lib(LIB, OBJ, [], force, verbose)
        binding.result()
    if force or _stale(MEASURE_LIB, [MEASURE_SRC, os.path.join(CSRC, "measure", "dfa3d_measure.h")]):
        _run([hipcc, *FLAGS, "-shared", MEASURE_SRC, "-o", MEASURE_LIB], verbose)
    if clocks:
        _build_lib(CLOCKS_LIB, os.path.join(OBJ, "clocks"), CLOCKS_FLAGS, force, verbose)
    return LIB


if __name__ == "__main__":
    build(force="--force" in sys.argv, clocks="--clocks" in sys.argv)
    print(LIB)
