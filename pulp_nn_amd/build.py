"""Compiles the HIP library for gfx950: one shared object per batch-norm width.

    python -m pulp_nn_amd.build          # both libraries
"""
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def lib_path(bn_bits):
    return os.path.join(LIBDIR, "libpulpnn_hip%d.so" % bn_bits)


# translation units of the library: the host layer with most kernels, and kernel families compiled beside it
UNITS = ("conv", "conv_band", "conv_rows", "pw_any", "dwpw", "depthwise", "dw_hwc", "dw_mfma", "pulp_nn_hip")


def _run(cmd, what, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # the host pass warns that it does not know the packed-fp32 feature: harmless
    log = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError("%s failed:\n" % what + log)
    if verbose and log.strip():
        print(log)


def compile_unit(bn_bits, unit, obj, verbose=False):
    _run([HIPCC] + FLAGS + ["-c", "-DPULPNN_BN_BITS=%d" % bn_bits, os.path.join(CSRC, unit + ".hip"), "-o", obj], "hipcc", verbose)
    return obj


def build(bn_bits, verbose=False, pool=None):
    """Compiles the units side by side (on `pool` if given) and links them into one shared object."""
    from concurrent.futures import ThreadPoolExecutor
    os.makedirs(LIBDIR, exist_ok=True)
    out = lib_path(bn_bits)
    with tempfile.TemporaryDirectory() as tmp, ThreadPoolExecutor(4) as own:
        jobs = [(pool or own).submit(compile_unit, bn_bits, u, os.path.join(tmp, u + ".o"), verbose) for u in UNITS]
        objs = [j.result() for j in jobs]
        _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", out], "link", verbose)
    return out


TOOLS = ("mfma_ceiling", "conv_phases", "hbm_ceiling")


def tool_path(name="mfma_ceiling"):
    return os.path.join(LIBDIR, name)


def build_tool(name="mfma_ceiling", verbose=False):
    """The measurement tools: the matrix-core yardstick (csrc/mfma_ceiling.hip) and the phase / ablation trace of
    the large convolution (csrc/conv_phases.hip), the plain-copy memory yardstick (csrc/hbm_ceiling.hip).  Stand-alone executables, no part of the libraries."""
    os.makedirs(LIBDIR, exist_ok=True)
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", os.path.join(CSRC, name + ".hip"), "-o", tool_path(name)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + res.stdout)
    return tool_path(name)


def fast_path():
    return os.path.join(LIBDIR, "_pulpnn_fast.so")


def tensor_path():
    return os.path.join(LIBDIR, "_pulpnn_tensor.so")


def build_fast(verbose=False):
    """The Python front end's call path, host code only: csrc/pybind_fast.cpp, a CPython extension module, and
    csrc/pybind_tensor.cpp, which knows torch's tensors."""
    import sysconfig
    from torch.utils import cpp_extension
    os.makedirs(LIBDIR, exist_ok=True)
    gxx = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-I", sysconfig.get_paths()["include"]]
    _run(gxx + [os.path.join(CSRC, "pybind_fast.cpp"), "-o", fast_path()], "g++", verbose)
    libs = cpp_extension.library_paths()
    _run(gxx + ["-I" + d for d in cpp_extension.include_paths()] + [os.path.join(CSRC, "pybind_tensor.cpp"), "-o", tensor_path()] +
         ["-L" + d for d in libs] + ["-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10"] + ["-Wl,-rpath," + d for d in libs], "g++", verbose)
    return fast_path()


def demo_path():
    return os.path.join(LIBDIR, "capi_demo")


def build_demo(verbose=False):
    """The plain C caller (csrc/capi_demo.c), compiled by gcc as C99 against include/ and linked with the 32-bit
    library: what a reference-side application's build does.  Needs libpulpnn_hip32.so to exist."""
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cmd = ["gcc", "-std=c99", "-O2", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(os.path.dirname(HERE), "include"),
           "-I", os.path.join(rocm, "include"), os.path.join(CSRC, "capi_demo.c"), "-o", demo_path(),
           "-L", LIBDIR, "-lpulpnn_hip32", "-L", os.path.join(rocm, "lib"), "-lamdhip64",
           "-Wl,-rpath,$ORIGIN", "-Wl,-rpath," + os.path.join(rocm, "lib")]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError("gcc failed:\n" + res.stdout)
    return demo_path()


def build_all(verbose=False):
    from concurrent.futures import ThreadPoolExecutor
    with ThreadPoolExecutor(2) as ex, ThreadPoolExecutor(6) as units:
        libs = [ex.submit(build, b, verbose, units) for b in (32, 64)]
        tools = [units.submit(build_fast, verbose)] + [units.submit(build_tool, t, verbose) for t in TOOLS]
        out = [f.result() for f in libs] + [f.result() for f in tools]
    return out + [build_demo(verbose)]


if __name__ == "__main__":
    for p in build_all(verbose=True):
        print("built", p)
