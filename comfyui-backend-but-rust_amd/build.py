"""Build libgpu_kernels.so (the C-ABI library of the gfx950 kernels) in-tree with hipcc.

hipcc cross-compiles for gfx950 without a GPU.  Objects are built in parallel, one per .hip file, then linked.
"""
import concurrent.futures
import glob
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libgpu_kernels.so")
ARCH = os.environ.get("HIP_ARCH", "gfx950")
SOURCES = ["quant_rows.hip", "prologue_rows.hip", "weight_formats.hip", "act_tables.hip", "int8_gemm.hip", "w6.hip", "w6_requant.hip", "w6a8_group_gemm.hip", "attn_int8.hip"]
FLAGS = [
    "--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    # exact arithmetic: no contraction except where fmaf is written, IEEE divide, no fast-math
    "-ffp-contract=off", "-fno-fast-math", "-fhip-fp32-correctly-rounded-divide-sqrt",
    # keep the compiler from forming packed-fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the DMA sequences name m0 as clobbered on purpose; the compiler remarks on every one
    "-Wno-inline-asm",
]
# Per-file additions.  The grouped W6A8 kernel reads every MFMA result with VALU instructions (int32 partial -> fp32),
# which cannot take accumulator registers as operands: keep its MFMA destinations in ordinary vector registers.
EXTRA = {"w6a8_group_gemm.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}


def _compile(src):
    obj = os.path.join(CSRC, os.path.splitext(src)[0] + ".o")
    cmd = ["hipcc", *FLAGS, *EXTRA.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (src, err))
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


BLAS_OUT = os.path.join(HERE, "libgpu_blas.so")


def build_blas():
    """The dense-GEMM library over hipBLASLt: host code only."""
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["hipcc", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
                           os.path.join(CSRC, "blas_gemm.cpp"), "-o", BLAS_OUT, "-L" + os.path.join(rocm, "lib"), "-lhipblaslt",
                           "-Wl,-rpath," + os.path.join(rocm, "lib")])
    return BLAS_OUT


def _torch():
    """torch for ROCm, or None: the libraries and ffi.py do without it."""
    try:
        import torch
    except ImportError:
        return None
    return torch if torch.version.hip else None


def calls_out():
    """The file of the native calls.  Its name carries the Python and the torch that it is compiled against: others look for another."""
    import torch
    return os.path.join(HERE, "_pycalls-torch" + torch.__version__ + sysconfig.get_config_var("EXT_SUFFIX"))


def drop_calls():
    """Native calls of any torch: compiled against a kernel library and header that are about to change."""
    for f in glob.glob(os.path.join(glob.escape(HERE), "_pycalls*.so")):
        os.remove(f)


def build_calls():
    """The Python calls that are native code (csrc/py_linear.cpp): host code only, against torch's headers and libgpu_kernels.so."""
    drop_calls()
    torch = _torch()
    if torch is None:
        sys.stderr.write("torch for ROCm cannot be imported: the native calls of the Python side (csrc/py_linear.cpp) are left out\n")
        return None
    out = calls_out()
    part = os.path.join(HERE, "_pycalls-unfinished.so")
    t, rocm = os.path.dirname(torch.__file__), os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                           "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI), "-isystem", os.path.join(t, "include"),
                           "-isystem", os.path.join(rocm, "include"), "-isystem", sysconfig.get_paths()["include"],
                           os.path.join(CSRC, "py_linear.cpp"), "-o", part, "-L" + os.path.join(t, "lib"), "-L" + HERE, "-lgpu_kernels",
                           "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-Wl,-rpath,$ORIGIN"])
    os.replace(part, out)
    return out


def _older(out, deps):
    return not os.path.exists(out) or any(os.path.getmtime(d) > os.path.getmtime(out) for d in deps)


def stale():
    """Whether an output is missing or older than what it is made from: each by its own time, since a later one's compilation may have failed."""
    include = os.path.join(os.path.dirname(HERE), "include")
    kernels = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".hpp"))] + [os.path.join(include, "gpu_api.h")]
    return (_older(OUT, kernels) or _older(BLAS_OUT, [os.path.join(CSRC, "blas_gemm.cpp"), os.path.join(include, "gpu_blas_api.h")]) or
            (_torch() is not None and _older(calls_out(), [os.path.join(CSRC, "py_linear.cpp"), os.path.join(include, "gpu_api.h"), OUT])))


def build(force=True):
    if not force and not stale():
        return OUT
    with concurrent.futures.ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
        objs = list(ex.map(_compile, SOURCES))
    drop_calls()
    subprocess.check_call(["hipcc", "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", OUT, *objs])
    build_blas()
    build_calls()
    return OUT


if __name__ == "__main__":
    print(build(force="--if-stale" not in sys.argv))
