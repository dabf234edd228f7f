"""Builds the C-ABI libraries with hipcc for gfx950: libe2h_quant.so (include/e2h_quant.h, the quantized linears and the
Llama decode step) and libe2h_seq.so (include/e2h_seq.h, the layers with per-sequence state and
mixtures of experts).

A third, small object is a CPython extension module: the host side of calls of small linears (_calls.so, csrc/e2h_calls.cpp).

The libraries are built in-tree, next to this file, so that they travel with the source tree; nothing is
installed into site-packages and no JIT cache is involved.  They are separate so that a model that needs one of them
compiles only that one.
"""

import os
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
LIB_PATH = PKG_DIR / "libe2h_quant.so"
SEQ_LIB_PATH = PKG_DIR / "libe2h_seq.so"
CALLS_PATH = PKG_DIR / "_calls.so"

SOURCES = ["e2h_abi.hip", "e2h_quantize.hip", "e2h_int4_mm.hip", "e2h_int4_staged.hip", "e2h_int4_staged_g32.hip", "e2h_int4_staged_g64.hip", "e2h_int4_staged_g128.hip", "e2h_int8_mm.hip", "e2h_int8_stream.hip", "e2h_int4_gemm.hip", "e2h_int4_gemm128.hip", "e2h_int8_gemm.hip", "e2h_unpacked_gemm.hip", "e2h_attention.hip", "e2h_sample.hip", "e2h_probe.hip"]

SEQ_SOURCES = ["e2h_seq_norm.hip", "e2h_seq_linear.hip", "e2h_seq_attention.hip", "e2h_seq_hgrn2.hip", "e2h_seq_delta.hip", "e2h_seq_moe.hip"]

# -ffp-contract=off: the quantizers are bit-exact restatements of separate torch ops; an FMA formed
# across two of them would change codes.  packed-fp32-ops is switched off because some packed float32
# forms have produced wrong results on the target machines.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fno-fast-math",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


# Per-source additions.  The 32x32-tile matmul mixes MFMA accumulators with float32 FMAs on the same values; with
# the accumulators in the accumulation register file every FMA needs copies in and out (3 extra instructions per FMA),
# so that file is compiled with MFMA results kept in ordinary vector registers.
_VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form"]
EXTRA_FLAGS = {s: _VGPR_FORM for s in ("e2h_int4_gemm.hip", "e2h_int4_staged_g32.hip", "e2h_int4_staged_g64.hip", "e2h_int4_staged_g128.hip")}  # (the int8 kernel of the same shape has no such FMAs)


def _hipcc():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found; the e2h kernels cannot be built")


def _run(cmd):
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(map(str, cmd)), proc.stdout))
    return proc.stdout


def _compile_and_link(names, lib_path, verbose):
    hipcc = _hipcc()
    obj_dir = PKG_DIR / "build"
    obj_dir.mkdir(exist_ok=True)
    sources = [s for s in names if (CSRC / s).exists()]

    def compile_one(src):
        obj = obj_dir / (Path(src).stem + ".o")
        out = _run([hipcc, *HIPCC_FLAGS, *EXTRA_FLAGS.get(src, []), "-c", str(CSRC / src), "-o", str(obj)])
        if verbose and out.strip():
            print(out)
        return obj

    with ThreadPoolExecutor(max_workers=min(len(sources), 6)) as pool:
        objs = list(pool.map(compile_one, sources))
    tmp = lib_path.with_name(lib_path.name + ".tmp")
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)])
    os.replace(tmp, lib_path)
    return lib_path


def build_library(verbose=False):
    """Compile every HIP source of libe2h_quant.so for gfx950 and link it.  Always recompiles."""
    return _compile_and_link(SOURCES, LIB_PATH, verbose)


def build_seq_library(verbose=False):
    """The same for libe2h_seq.so."""
    return _compile_and_link(SEQ_SOURCES, SEQ_LIB_PATH, verbose)


def build_calls(verbose=False):
    """The host-side extension module of small calls (csrc/e2h_calls.cpp), for the installed torch and no other."""
    import sysconfig

    import torch

    home = Path(torch.__file__).resolve().parent
    rocm = Path(_hipcc()).resolve().parent.parent
    cxx = shutil.which(os.environ.get("CXX", "g++")) or rocm / "llvm" / "bin" / "clang++"  # else the one that hipcc drives
    tmp = CALLS_PATH.with_name(CALLS_PATH.name + ".tmp")
    out = _run([cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
                f'-DE2H_TORCH_VERSION="{torch.__version__}"',
                *(f"-I{d}" for d in (home / "include", home / "include" / "torch" / "csrc" / "api" / "include", rocm / "include", sysconfig.get_paths()["include"])),
                str(CSRC / "e2h_calls.cpp"), "-o", str(tmp), f"-L{home / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python"])
    if verbose and out.strip():
        print(out)
    os.replace(tmp, CALLS_PATH)
    return CALLS_PATH


if __name__ == "__main__":
    print(build_library(verbose=True))
    print(build_seq_library(verbose=True))
    print(build_calls(verbose=True))
