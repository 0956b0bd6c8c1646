"""CPU-only checks of the drop-in boundary: the library loads, exports every symbol the header declares, and refuses bad
arguments with the reference's return codes before touching the GPU."""
import ctypes
import json
import os
import re
import subprocess

import numpy as np
import pytest

import oracle
from conftest import ROOT, pkg

ffi = pkg("ffi")


def header_functions(name="gpu_api.h"):
    text = open(os.path.join(ROOT, "include", name)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return re.findall(r"\b(gpu_[a-z0-9_]+)\s*\(", text)


def test_library_exports_every_declared_symbol():
    names = header_functions()
    assert {"gpu_quant_rows", "gpu_quant_rows_b", "gpu_rotate_rows_f32", "gpu_sd_quant_rows", "gpu_int8_gemm",
            "gpu_int8_gemm_residual", "gpu_w6_decode"} <= set(names)
    lib = ctypes.CDLL(ffi.LIB_PATH)
    for n in names:
        assert hasattr(lib, n), n
    for n in ffi.SIGNATURES:
        assert n in names, "ffi.py binds %s, which the header does not declare" % n
    assert "gfx950" in ffi.build_info()
    # the dense-GEMM library: loads (hipBLASLt resolves) and exports what its header declares
    blas_names = header_functions("gpu_blas_api.h")
    assert set(blas_names) == {"gpu_blas_init", "gpu_gemm"} == set(ffi.BLAS_SIGNATURES)
    blas = ctypes.CDLL(ffi.BLAS_LIB_PATH)
    for n in blas_names:
        assert hasattr(blas, n), n
    assert ffi.blas().gpu_gemm(0, 0, 0, 0, 0, 0, 0, 4, 4, 4, 1, 2, 2, 1.0, 0.0, 0) == -100    # before gpu_blas_init


def test_header_constants_match_reference_codes():
    text = open(os.path.join(ROOT, "include", "gpu_api.h")).read()
    assert re.search(r"DT_F32 = 0, DT_F16 = 1, DT_BF16 = 2", text)
    assert (ffi.PRO_PLAIN, ffi.PRO_RMS, ffi.PRO_GATE, ffi.PRO_SWIGLU, ffi.PRO_ADALN, ffi.PRO_SITU_FAST) == (0, 1, 2, 3, 7, 13)
    for name, val in (("PRO_LN_MOD", 9), ("PRO_LN_AFFINE", 10), ("PRO_GELU_TANH", 11), ("PRO_LN_AFFINE_SILU", 12)):
        assert re.search(r"%s = %d\b" % (name, val), text)


def q(dtype=2, pro=0, K=256, rotate=0, M=4):
    return ffi.raw("gpu_quant_rows", dtype, pro, 0, K, 0, 0, 0, 0, 0.0, 0, 0, 0, 0, M, K, rotate, 0)


def test_quant_rows_refusals_match_reference_order():
    assert q(K=200) == -1                       # csrc/kernels.cu:275
    assert q(K=320, rotate=1) == -1
    assert q(K=192, rotate=128) == -1
    assert q(dtype=1) == -4                     # :297
    assert q(dtype=1, pro=99) == -4             # dtype is looked at before the prologue id
    assert q(pro=99) == -3 and q(pro=12) == -3  # :292 (LN_AFFINE_SILU is not in the quantizer's list)
    assert q(K=32768 + 256) == -2               # :265
    assert q(pro=ffi.PRO_SITU, M=0) == 0 and q(pro=ffi.PRO_SITU_FAST, M=0) == 0
    assert q(pro=ffi.PRO_RMS, M=0) == 0
    assert q(M=0) == 0
    # the oracle agrees on the shared codes
    x = np.zeros((1, 512), np.uint16)
    assert oracle.quant_rows(oracle.BF16, x, 200, 0)[0] == -1
    assert oracle.quant_rows(oracle.F16, x, 256, 0)[0] == -4


def test_other_entry_point_refusals():
    assert ffi.raw("gpu_quant_rows_b", 2, ffi.PRO_LN_MOD, 0, 300, 0, 0, 0.0, 0, 0, 0, 0, 1, 300, 0, 0) == -1
    assert ffi.raw("gpu_quant_rows_b", 0, ffi.PRO_LN_MOD, 0, 256, 0, 0, 0.0, 0, 0, 0, 0, 1, 256, 0, 0) == -4
    assert ffi.raw("gpu_quant_rows_b", 2, ffi.PRO_RMS, 0, 256, 0, 0, 0.0, 0, 0, 0, 0, 1, 256, 0, 0) == -3
    assert ffi.raw("gpu_rotate_rows_f32", ffi.PRO_PLAIN, 0, 320, 0, 0, 0.0, 0, 1, 320, 0) == -1
    assert ffi.raw("gpu_rotate_rows_f32", ffi.PRO_GATE, 0, 256, 0, 0, 0.0, 0, 1, 256, 0) == -3
    pr = lambda dt, pro: ffi.raw("gpu_prologue_rows", dt, pro, 0, 256, 0, 0, 0, 0, 0.0, 0, 0, 0, 256, 0, 256, 0)
    assert pr(1, ffi.PRO_RMS) == -4 and pr(2, ffi.PRO_LN_MOD) == -3 and pr(2, 99) == -3 and pr(2, ffi.PRO_RMS) == 0
    pb = lambda dt, pro: ffi.raw("gpu_prologue_rows_b", dt, pro, 0, 256, 0, 0, 0.0, 0, 0, 0, 256, 0, 256, 0)
    assert pb(7, ffi.PRO_LN_MOD) == -4 and pb(1, ffi.PRO_RMS) == -3 and pb(1, ffi.PRO_GELU_TANH) == 0
    assert ffi.raw("gpu_sd_quant_rows", 0, 640, 0, 0, 1, 640, 128, 0) == -1     # csrc/sd.cu:600
    assert ffi.raw("gpu_sd_quant_rows", 0, 640, 0, 0, 1, 640, 256, 0) == -1
    assert ffi.raw("gpu_w6_decode", 0, 0, 0, 4, 48, 32, 0) == -1                # csrc/h3.cu:41
    assert ffi.raw("gpu_w6_decode", 0, 0, 0, 4, 64, 8, 0) == -1
    assert ffi.raw("gpu_w6_decode", 0, 0, 0, 0, 64, 32, 0) == 0


def test_gemm_refusals_and_empty_shapes():
    g = lambda M, N, K, dt=2: ffi.raw("gpu_int8_gemm", 0, 0, 0, 0, 0, 0, M, N, K, dt, 0)
    assert g(0, 8, 16) == 0 and g(8, 0, 16) == 0 and g(8, 8, 0) == 0       # csrc/vendor/cutlass_gemm_int8.cu:377
    assert g(8, 8, 16, dt=5) == -200                                         # csrc/gemm.cu:126
    assert g(8, 8, 20) == -200                                               # K % 8: no tile configuration takes it (:191, :237-247)
    r = lambda M, N, K, rs=1, res=1, dt=2: ffi.raw("gpu_int8_gemm_residual", 0, 0, 0, 0, 0, rs, res, 0, M, N, K, dt, 0)
    assert r(0, 8, 16) == 0 and r(8, 0, 16) == 0                             # :353
    assert r(8, 8, 0) == -201                                                # :355, csrc/gemm.cu:137
    assert r(8, 8, 16, rs=0) == -201 and r(8, 8, 16, res=0) == -201          # :357
    assert r(8, 8, 16, dt=9) == -201


def test_ok_and_k_raise_like_the_reference():
    ffi.ok(0, "anything")
    with pytest.raises(ffi.KernelError, match="gpu_quant_rows failed with code -1"):
        ffi.k("gpu_quant_rows", 2, 0, 0, 200, 0, 0, 0, 0, 0.0, 0, 0, 0, 0, 4, 200, 0, 0)
    with pytest.raises(ffi.KernelError, match="x failed: "):
        ffi.ok(1, "x")


def test_oracle_reproduces_golden_fixtures(synth):
    import hashlib
    dig = lambda a: hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest()
    g = json.load(open(os.path.join(ROOT, "tests", "golden", "config0_w8a8.json")))
    c = synth.config0(0)
    assert dig(c["x"]) == g["x_sha256"] and dig(c["W"]) == g["W_sha256"] and dig(c["ws"]) == g["ws_sha256"]
    rc, qq, xs = oracle.quant_rows(oracle.BF16, c["x"], c["K"], 0)
    acc = oracle.int8_gemm_acc(qq, c["W"])
    assert dig(qq) == g["q_sha256"] and dig(xs.view(np.uint32)) == g["xs_bits_sha256"] and dig(acc) == g["acc_sha256"]
    assert qq.reshape(-1)[::g["stride"]].tolist() == g["q_sample"]
    d = oracle.epilogue(acc, xs, c["ws"], c["bias"], oracle.BF16, fma=1)
    assert dig(d) == g["d_fma_bits_sha256"] and d.reshape(-1)[::g["stride"]].tolist() == g["d_fma_bits_sample"]
    # the plain formula of the config text (scale = absmax/127, RNE, float product) lands within 1 code of the bf16 path
    x = synth.bf16_to_f32(c["x"])
    plain = np.clip(np.rint(x / (np.abs(x).max(1, keepdims=True) / np.float32(127))), -127, 127)
    assert np.abs(plain - qq).max() <= 1
    r = json.load(open(os.path.join(ROOT, "tests", "golden", "rotated_quant.json")))
    xr = synth.bf16_bits(synth.activations(11, 8, 1024, "t3"))
    assert dig(xr) == r["x_sha256"]
    for grp in (64, 128, 256):
        rc, q2, s2 = oracle.quant_rows(oracle.BF16, xr, 1024, grp)
        assert dig(q2) == r["q_g%d_sha256" % grp] and dig(s2.view(np.uint32)) == r["xs_bits_g%d_sha256" % grp]


def _write_checkpoint(path, extra=None, groupsize=256, scalar_scale=False):
    import torch
    from safetensors.torch import save_file
    g = torch.Generator().manual_seed(3)
    N, K = 64, 512
    t = {
        "blk.fc.weight": torch.randint(-127, 128, (N, K), dtype=torch.int8, generator=g),
        "blk.fc.weight_scale": torch.tensor([0.01]) if scalar_scale else torch.rand(N, generator=g) * 0.01 + 0.001,
        "blk.fc.bias": (torch.randn(N, generator=g) * 0.02).to(torch.bfloat16),
        "blk.fc.comfy_quant": torch.tensor(list(json.dumps({"format": "int8_tensorwise", "convrot": True,
                                                            "convrot_groupsize": groupsize}).encode()), dtype=torch.uint8),
        "blk.w6.weight": torch.randint(0, 256, (N, K * 3 // 4), dtype=torch.uint8, generator=g),
        "blk.w6.weight_s_rel": torch.randint(0x30, 0x50, (N, K // 32), dtype=torch.uint8, generator=g).view(torch.float8_e4m3fn),
        "blk.w6.weight_s_channel": torch.rand(N, generator=g) * 0.01,
        "blk.dense.weight": torch.randn(N, K, generator=g).to(torch.bfloat16),
    }
    t.update(extra or {})
    save_file(t, path)
    return t


def test_checkpoint_layouts_are_read_like_the_reference(tmp_path):
    import torch
    from safetensors import safe_open
    wts = pkg("weights")
    p = str(tmp_path / "a.safetensors")
    t = _write_checkpoint(p)
    with safe_open(p, framework="pt") as st:
        fc = wts.load_linear(st, "blk.fc", device="cpu")
        assert fc.kind == "int8_convrot" and (fc.n, fc.k) == (64, 512) and fc.scale.shape == (64,)
        assert torch.equal(fc.weight, t["blk.fc.weight"]) and fc.bias.dtype == torch.bfloat16
        w6 = wts.load_linear(st, "blk.w6", device="cpu")
        assert w6.kind == "w6" and (w6.n, w6.k) == (64, 512) and w6.s_rel.dtype == torch.uint8 and w6.s_rel.shape == (64, 16)
        assert wts.load_linear(st, "blk.dense", device="cpu").kind == "dense"
    # one scale for all rows is expanded on the host (src/relayvsr.rs:141-149)
    p2 = str(tmp_path / "b.safetensors")
    _write_checkpoint(p2, scalar_scale=True)
    with safe_open(p2, framework="pt") as st:
        s = wts.load_linear(st, "blk.fc", device="cpu").scale
        assert s.shape == (64,) and (s == s[0]).all()
    # other group sizes and scale counts are refused
    p3 = str(tmp_path / "c.safetensors")
    _write_checkpoint(p3, groupsize=64)
    with safe_open(p3, framework="pt") as st:
        with pytest.raises(wts.CheckpointError, match="groups of 256"):
            wts.load_linear(st, "blk.fc", device="cpu")
    p4 = str(tmp_path / "d.safetensors")
    _write_checkpoint(p4, extra={"blk.fc.weight_scale": torch.ones(7)})
    with safe_open(p4, framework="pt") as st:
        with pytest.raises(wts.CheckpointError, match="7 weight scales for 64 rows"):
            wts.load_linear(st, "blk.fc", device="cpu")


def test_makefile_and_build_script_list_the_same_units_and_flags():
    """The Makefile (native hosts) and build.py (this repository's Python side) must compile the same units with the
    same arithmetic flags, or the two libraries would differ in bits."""
    import importlib
    pkg_dir = os.path.join(ROOT, "comfyui-backend-but-rust_amd")
    mk = open(os.path.join(pkg_dir, "Makefile")).read()
    units = re.search(r"^UNITS\s*:=\s*(.+)$", mk, re.M).group(1).split()
    build = importlib.import_module("comfyui-backend-but-rust_amd.build")
    assert sorted(u + ".hip" for u in units) == sorted(build.SOURCES)
    flags = re.search(r"^FLAGS\s*:=\s*((?:.*\\\n)*.*)$", mk, re.M).group(1).replace("\\\n", " ").split()
    flags = [f.replace("$(ARCH)", build.ARCH) for f in flags]
    assert sorted(flags) == sorted(build.FLAGS)
    for src, extra in build.EXTRA.items():
        line = re.search(r"^csrc/%s\.o: FLAGS \+= (.+)$" % re.escape(src[:-4]), mk, re.M)
        assert line and line.group(1).split() == extra


def test_make_builds_the_libraries_without_python():
    """The default target is for hosts that link the kernels natively: nothing in it runs Python or needs torch."""
    out = subprocess.check_output(["make", "-n", "-B", "-C", os.path.join(ROOT, "comfyui-backend-but-rust_amd")], text=True)
    assert "libgpu_kernels.a" in out and "libgpu_kernels.so" in out and "libgpu_blas.so" in out
    assert "python" not in out and "py_linear" not in out


@pytest.mark.parametrize("torch", ["absent", "not for ROCm"])
def test_build_script_without_torch(torch, tmp_path, monkeypatch, capsys):
    """ctypes callers need no torch: without it the build script makes the libraries, and leaves out what only torch's users import."""
    import sys
    import types
    build = pkg("build")
    made = []
    other = types.SimpleNamespace(version=types.SimpleNamespace(hip=None), __file__="torch/__init__.py", _C=types.SimpleNamespace(_GLIBCXX_USE_CXX11_ABI=True))
    monkeypatch.setitem(sys.modules, "torch", None if torch == "absent" else other)   # None: import torch raises ImportError
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build, "_compile", lambda src: made.append(src) or src[:-4] + ".o")
    monkeypatch.setattr(build.subprocess, "check_call", lambda cmd: made.append(cmd[cmd.index("-o") + 1]))
    assert build.build() == build.OUT
    assert made[-2:] == [build.OUT, build.BLAS_OUT] and sorted(made[:-2]) == sorted(build.SOURCES)
    assert "torch" in capsys.readouterr().err


def test_build_script_knows_which_outputs_are_older_than_their_sources(tmp_path, monkeypatch):
    """Every output against its own sources: a compilation that failed behind the kernel library's leaves an old file that is not
    taken for a new one, nor is one that was compiled against another torch or Python."""
    build = pkg("build")
    csrc, include = tmp_path / "pkg" / "csrc", tmp_path / "include"
    csrc.mkdir(parents=True)
    include.mkdir()
    monkeypatch.setattr(build, "HERE", str(tmp_path / "pkg"))
    monkeypatch.setattr(build, "CSRC", str(csrc))
    for name in ("OUT", "BLAS_OUT"):
        monkeypatch.setattr(build, name, str(tmp_path / "pkg" / os.path.basename(getattr(build, name))))
    calls = build.calls_out()
    sources = [csrc / "quant_rows.hip", csrc / "common.hpp", csrc / "blas_gemm.cpp", csrc / "py_linear.cpp", include / "gpu_api.h", include / "gpu_blas_api.h"]

    def touch(path, when):
        open(path, "a").close()
        os.utime(path, (when, when))

    def tree(**later):   # sources at 100, the libraries at 200, the native calls, linked against the first of them, at 210
        for p in sources:
            touch(p, later.get(p.name.replace(".", "_"), 100))
        touch(build.OUT, later.get("out", 200))
        touch(build.BLAS_OUT, later.get("blas", 200))
        touch(calls, later.get("calls", 210))
        return build.stale()

    assert not tree()
    assert tree(py_linear_cpp=220) and tree(blas_gemm_cpp=220) and tree(common_hpp=220) and tree(quant_rows_hip=220) and tree(gpu_api_h=220)
    # the kernel library was linked anew, and then the other compilation failed
    assert tree(py_linear_cpp=220, out=230, blas=230) and tree(gpu_api_h=220, out=230, blas=230)
    assert tree(blas_gemm_cpp=220, out=230, calls=240) and tree(out=230, blas=230)
    assert not tree(py_linear_cpp=220, out=230, blas=230, calls=240)
    import torch
    monkeypatch.setattr(torch, "__version__", "0.0.1")
    assert build.stale()


def test_build_script_leaves_no_old_native_calls_behind_a_failure(tmp_path, monkeypatch):
    """What was compiled against the former kernel library is gone before the new one is there, and a file appears whole."""
    build = pkg("build")
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    for name in ("OUT", "BLAS_OUT"):
        monkeypatch.setattr(build, name, str(tmp_path / os.path.basename(getattr(build, name))))
    calls = build.calls_out()
    open(calls, "w").close()
    monkeypatch.setattr(build, "_compile", lambda src: src[:-4] + ".o")

    def run(cmd):
        out = cmd[cmd.index("-o") + 1]
        assert out != calls and not os.path.exists(calls)
        if cmd[0] == "g++":
            open(out, "w").close()
            raise subprocess.CalledProcessError(1, cmd)

    monkeypatch.setattr(build.subprocess, "check_call", run)
    with pytest.raises(subprocess.CalledProcessError):
        build.build()
    assert not os.path.exists(calls)


def _package_with(tmp_path, native):
    """The package beside its kernel library in a folder of its own, its native calls as `native` makes them; what a process that imports
    qlinear from there prints or fails with."""
    import sys
    src = os.path.join(ROOT, "comfyui-backend-but-rust_amd")
    dst = tmp_path / "comfyui-backend-but-rust_amd"
    dst.mkdir()
    for f in os.listdir(src):
        if f.endswith(".py") or f in ("libgpu_kernels.so", "libgpu_blas.so"):
            os.symlink(os.path.join(src, f), dst / f)
    native(dst)
    code = """if True:
        import importlib
        ql = importlib.import_module("comfyui-backend-but-rust_amd.qlinear")
        ql._linear_w8a8 = lambda *args: args
        print(ql._pycalls, ql.linear_w8a8(1, 2, 3, rotate=64))
    """
    return subprocess.run([sys.executable, "-c", code], cwd=tmp_path, capture_output=True, text=True, timeout=300)


def test_qlinear_without_the_native_calls(tmp_path):
    """A tree with the kernel library alone: qlinear is there, and its calls are made in Python."""
    r = _package_with(tmp_path, lambda d: None)
    assert r.returncode == 0 and r.stdout.split("\n")[0] == "None (1, 2, 3, None, 64, None)", r.stderr[-500:]


def test_qlinear_names_the_build_where_the_native_calls_do_not_load(tmp_path):
    """A file that is there and cannot be loaded is an error that says what to run, not a reason to run slower."""
    name = os.path.basename(pkg("build").calls_out())
    r = _package_with(tmp_path, lambda d: (d / name).write_bytes(b"no library"))
    assert r.returncode != 0 and "ImportError" in r.stderr and "build.py" in r.stderr and name in r.stderr, r.stderr[-500:]


def test_rust_host_crate_follows_the_headers_and_the_build_script():
    """rust/src/sys.rs is generated from the headers (same names, arity and scalar types as the ctypes table), and
    rust/build.rs compiles the units and flags that build.py does.  No Rust toolchain is needed for either check."""
    import importlib
    import subprocess
    import sys
    r = subprocess.run([sys.executable, os.path.join(ROOT, "rust", "gen_sys.py"), "--check"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    text = open(os.path.join(ROOT, "rust", "src", "sys.rs")).read()
    decls = {m.group(1): m.group(2) for m in re.finditer(r"pub fn (gpu_\w+)\(([^)]*)\)", text)}
    assert set(decls) == set(header_functions()) | set(header_functions("gpu_blas_api.h"))
    # c_uint64 and c_size_t are one ctypes class on this platform
    kinds = {ffi._P: {"P", "PM"}, ffi._I64: {"i64"}, ffi._I32: {"i32"}, ffi._F32: {"f32"}, ffi._U64: {"u64", "usize"}}
    for table in (ffi.SIGNATURES, ffi.BLAS_SIGNATURES):
        for name, argtypes in table.items():
            rust = [a.split(":")[1].strip() for a in " ".join(decls[name].split()).split(",") if a.strip()]
            assert len(rust) == len(argtypes), name
            for rt, ct in zip(rust, argtypes):
                assert rt in kinds[ct], (name, rt, ct)
    build = importlib.import_module("comfyui-backend-but-rust_amd.build")
    rs = open(os.path.join(ROOT, "rust", "build.rs")).read()
    units = re.findall(r'"(\w+\.hip)"', rs[rs.index("const UNITS"):rs.index("];")])
    assert sorted(units) == sorted(build.SOURCES)
    for flag in build.FLAGS:
        if not flag.startswith("--offload-arch"):
            assert '"%s"' % flag in rs, flag
    for src, extra in build.EXTRA.items():
        assert src in rs and all('"%s"' % e in rs for e in extra)


KEPT_BUFFERS = r"""
#include "kept_buffers.hpp"
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
static KeptBuffers<2> kept;
static std::mutex queue_mu;
static std::vector<int> queue_;   // thread * 2 + launch
static char memory[4][64];
static int made = 0;
int main() {
    const auto make = [](size_t) -> void* { return memory[made++]; };
    const auto call = [&](int thread) {
        for (int i = 0; i < 20; ++i)
            kept.with(0, nullptr, 8, 64, make, [&](void*) {
                for (int launch = 0; launch < 2; ++launch) {
                    { std::lock_guard<std::mutex> lock(queue_mu); queue_.push_back(thread * 2 + launch); }
                    std::this_thread::sleep_for(std::chrono::microseconds(300));
                }
            });
    };
    std::thread a(call, 0), b(call, 1);
    a.join();
    b.join();
    if (queue_.size() != 80 || made != 1) return 1;
    for (size_t i = 0; i < queue_.size(); i += 2)
        if (queue_[i] % 2 != 0 || queue_[i + 1] != queue_[i] + 1) return 2;   // a call's launches stand together
    // one buffer per (device, stream); none where the call needs more than it holds, where it cannot be made, or beyond the last
    int other = 0;
    void *p0 = nullptr, *p1 = nullptr;
    const auto none = [](size_t) -> void* { return nullptr; };
    const auto ignore = [](void*) {};
    if (kept.with(0, nullptr, 65, 64, make, ignore) || kept.with(0, &other, 65, 64, make, ignore)) return 3;
    if (kept.with(0, &other, 8, 64, none, ignore) || made != 1) return 4;
    if (!kept.with(0, nullptr, 64, 64, make, [&](void* p) { p0 = p; }) || !kept.with(0, &other, 8, 64, make, [&](void* p) { p1 = p; })) return 5;
    if (p0 != memory[0] || p1 != memory[1] || made != 2) return 6;
    if (kept.with(1, nullptr, 8, 64, make, ignore) || made != 2) return 7;
    std::puts("ok");
    return 0;
}
"""


def test_calls_of_two_threads_on_one_stream_keep_their_launches_together(tmp_path):
    """The buffer that a split-K GEMM's two launches share: what a second thread queues on the same stream comes before or behind
    both of them, never between."""
    src, exe = tmp_path / "kept.cpp", str(tmp_path / "kept")
    src.write_text(KEPT_BUFFERS)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "comfyui-backend-but-rust_amd", "csrc"), str(src), "-o", exe])
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout)


def gemm_plan(M, N, K, start=0, aligned=1):
    out = (ctypes.c_int32 * 3)()
    assert ffi.raw("gpu_internal_int8_gemm_plan", M, N, K, start, aligned, ctypes.cast(out, ctypes.c_void_p)) == 0
    return tuple(out)


def test_gemm_operands_off_16_bytes_keep_the_kernels_that_take_them():
    """The kernel for up to 128 rows takes operands from 16-byte addresses only, the other two with DMA from 4-byte ones; and off 16
    bytes those run the sizes from which they always did, the register-staged tiles what is smaller."""
    def fetches(M, N, K):   # off 16 bytes, a multiple of 4
        tiles = -(-M // 128) * -(-N // 192)
        if K % 128:
            return False
        if M <= 256 and N >= 1024 and K >= 512:
            return K >= 1536 or (M > 128 and N >= 8192)
        if M >= 512 and N >= 512 and tiles > 256:
            return True
        return M > 128 and N >= 192 and (tiles >= 96 or (tiles >= 40 and K >= 2048) or (M <= 512 and N >= 1024 and K >= 8192))

    assert gemm_plan(64, 136, 384)[0] == 7 and gemm_plan(4608, 12288, 3072)[0] == 9   # 16-byte starts: everything but the smallest
    taken = set()
    for M in (1, 3, 64, 128, 129, 256, 300, 512, 2048, 8192):
        for N in (8, 136, 192, 512, 640, 1024, 4096, 8192, 12288):
            for K in (64, 128, 384, 512, 1024, 1536, 2048, 8192):
                for start in range(1, 16):
                    family = gemm_plan(M, N, K, start)[0]
                    if start % 4 == 0 and fetches(M, N, K):
                        assert family in (7, 9), (M, N, K, start)
                    else:
                        assert family in (1, 2), (M, N, K, start, family)
                    taken.add(family)
    assert taken == {1, 2, 7, 9}


def test_gemm_choice_where_it_was_measured():
    """Shapes at which one kernel, or another number of slices of K, was timed at least 8 % faster than the others with weights from HBM."""
    for M, N, K in [(1, 5120, 2048), (16, 8192, 2048), (4, 1280, 4096), (17, 3072, 3072), (32, 2048, 3072), (64, 2048, 2048), (48, 5120, 3072), (64, 640, 5120), (1, 12552, 3968), (1, 10240, 5120), (20, 7520, 6144), (17, 7304, 13312), (21, 5384, 7808),
                    (41, 7376, 3712), (44, 5184, 3840), (56, 7816, 4992), (35, 7880, 9216), (11, 15688, 13312)]:
        assert gemm_plan(M, N, K)[0] == 5, (M, N, K)
    for M, N, K in [(8, 4096, 640), (16, 24576, 4096), (17, 9216, 2048), (22, 3072, 6144), (35, 2952, 4224), (41, 1760, 4224), (60, 4096, 8192), (64, 1280, 2560), (65, 1280, 2048), (128, 4096, 3072)]:
        assert gemm_plan(M, N, K)[0] == 7, (M, N, K)
    for M, N, K in [(128, 3072, 5120), (96, 640, 2560), (256, 1280, 5120), (256, 8448, 12288), (512, 640, 5120), (1024, 320, 5120)]:
        family, _, slices = gemm_plan(M, N, K)
        assert family == 7 and slices > 1, (M, N, K, slices)
    for M, N, K in [(96, 24576, 8192), (256, 24576, 4096), (8192, 640, 2560), (2048, 1280, 1280), (1024, 4096, 2560)]:
        family, _, slices = gemm_plan(M, N, K)
        assert family == 7 and slices == 1, (M, N, K, slices)
    for M, N, K in [(4608, 3072, 3072), (8192, 5120, 640), (1024, 9216, 4096), (5366, 3144, 128)]:
        assert gemm_plan(M, N, K)[0] == 9, (M, N, K)


def test_gemm_store_policy_where_it_was_measured():
    """16-bit outputs of 40 to 100 MB: rows of whole 64 bytes are written through the L2 (by the default policy up to 1.13 times as long), others by
    the default policy (past the caches up to 1.8 times as long, written through 1.4)."""
    for M, N, K, policy in [(8192, 5120, 640, 1), (4096, 10240, 1280, 1), (4420, 4864, 1024, 1), (4160, 6144, 256, 1), (6154, 4896, 256, 1),
                            (5114, 4976, 256, 2), (8192, 5128, 640, 2), (7807, 3088, 256, 2), (6385, 7000, 256, 2),
                            (3655, 5376, 768, 0), (4608, 12288, 3072, 0), (8192, 8192, 512, 0), (3000, 5000, 768, 0)]:   # too small, too large
        assert gemm_plan(M, N, K)[:2] == (9, policy), (M, N, K)


def test_gemm_choice_for_32_bit_outputs():
    """Shapes of which the other kernel took 8 % and more longer: with 32-bit outputs, one round of 128-row tiles and short K, the one with
    fetching waves is the faster one; with longer K or several rounds it is not."""
    for M, N, K in [(5377, 1112, 768), (7465, 840, 384), (2433, 2648, 768), (2482, 2360, 256), (3159, 2104, 256), (5599, 1128, 768)]:
        assert gemm_plan(M, N, K, aligned=3)[0] == 7, (M, N, K)
    for M, N, K in [(4608, 12288, 3072), (817, 9176, 8704), (1423, 4240, 1792), (8192, 5120, 640)]:
        assert gemm_plan(M, N, K, aligned=3)[0] == 9, (M, N, K)
    for M in (512, 1030, 2433, 5377, 8192):   # 32-bit outputs change nothing else
        for N in (512, 840, 1112, 2648, 5120, 12288):
            for K in (256, 768, 1024, 1152, 4096):
                narrow, wide = gemm_plan(M, N, K), gemm_plan(M, N, K, aligned=3)
                tiles = -(-M // 128) * -(-N // 256)
                assert narrow[0] == wide[0] or (tiles <= 256 and K <= 1024 and (narrow[0], wide[0]) == (9, 7)), (M, N, K)


@pytest.mark.parametrize("b,h,lq,lk,d,shared", [(2, 9, 492, 492, 128, False), (1, 20, 516, 516, 128, False), (1, 19, 602, 602, 64, False), (2, 11, 356, 560, 128, False),
                                                (1, 21, 686, 686, 64, False), (1, 11, 640, 640, 128, False), (2, 6, 1029, 539, 64, False), (1, 2, 1849, 877, 128, True),
                                                (2, 15, 300, 1859, 64, True), (1, 10, 1024, 1024, 128, True), (1, 24, 4608, 4608, 128, True), (2, 10, 4096, 4096, 64, True)])
def test_attention_shares_keys_where_that_was_measured_faster(b, h, lq, lk, d, shared):
    """A workspace that ends with the column sums of V has no room for parts: no row block's keys are shared."""
    out = (ctypes.c_int64 * 10)()
    assert ffi.raw("gpu_internal_attn_layout_d", b, h, h, lq, lk, d, ctypes.cast(out, ctypes.c_void_p)) == 0
    vsum, kb = out[7], out[9]
    plain = vsum + (b * h * kb * d * 4 + 255) // 256 * 256
    total = ffi.lib.gpu_int8_attn_workspace_d(b, h, h, lq, lk, d)
    assert (total > plain) == shared and total >= plain


def test_w6_requant_rows_of_a_workgroup_where_they_were_measured():
    """Row counts that took 5 % and more off the other choices."""
    for N, K, rows in [(448, 2048, 2), (318, 2048, 2), (405, 1792, 2), (299, 4864, 2), (453, 5120, 2), (5376, 5376, 3), (4096, 1280, 4), (8192, 256, 4), (4096, 1536, 2), (4096, 7680, 1)]:
        assert ffi.raw("gpu_internal_w6_requant_rows", N, K) == rows, (N, K)
    for N in (1, 64, 300, 1000, 2276, 3127, 12288, 24576):
        for K in range(256, 39680 + 1, 256):
            rows = ffi.raw("gpu_internal_w6_requant_rows", N, K)
            assert 1 <= rows <= 16 and (rows == 1 or rows * K <= 16384), (N, K, rows)   # what its LDS array and 16 waves hold
    assert ffi.raw("gpu_internal_w6_requant_rows", 4, 300) == -1
