"""Build libtkm_attn.so: the HIP attention kernels for gfx950, the C ABI of include/tkm_attn.h
and include/tkm_prep.h, and the C host code that generates, compiles (hipRTC) and launches the
qkv-prep kernels.

Usage: python -m tokamak_amd.build   (or build() from Python).  Always recompiles.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
INCLUDE = os.path.join(ROOT, "include")
LIB_NAME = "libtkm_attn.so"
LIB_PATH = os.path.join(PKG, LIB_NAME)
# The runtime library: everything of libtkm_attn.so plus the tkm.h runtime (tkm_hip.c), the
# whole-graph generator, the hipBLASLt GEMMs and the runtime's kernels.
HIP_LIB_PATH = os.path.join(PKG, "libtkm_hip.so")
RT_SOURCES = ["tkm_gemm.hip", "tkm_gemm_mfma.hip", "tkm_rt_kernels.hip"]
RT_C_SOURCES = ["tkm_codegen_hip.c", "tkm_hip.c"]
SOURCES = ["attn_fwd.hip", "attn_asm.hip", "attn_bwd.hip", "tkm_attn_abi.hip"]
# Hand-scheduled assembly kernels: (generator module, kernel symbol).  Each is generated,
# assembled for gfx950 and embedded in the library as a code object (a C byte array).
ASM_KERNELS = [("tokamak_amd.asmgen.attn_fwd", "tkm_fa_fwd_d128_f16"),
               ("tokamak_amd.asmgen.attn_fwd", "tkm_fa_fwd_d128_bf16"),
               ("tokamak_amd.asmgen.attn_dkdv", "tkm_fa_bwd_dkdv_d128_f16"),
               ("tokamak_amd.asmgen.attn_dkdv", "tkm_fa_bwd_dkdv_d128_bf16"),
               ("tokamak_amd.asmgen.attn_dq", "tkm_fa_bwd_dq_d128_f16"),
               ("tokamak_amd.asmgen.attn_dq", "tkm_fa_bwd_dq_d128_bf16")]
C_SOURCES = ["tkm_error.c", "tkm_prelude.c", "tkm_codegen_util.c", "tkm_prep_codegen.c", "tkm_rtc.c",
             "tkm_plasma_codegen.c", "tkm_plasma_rt.c"]
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
ARCH = "gfx950"

# -packed-fp32-ops: no v_pk_{add,mul,fma}_f32 in generated code.
HIPFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", f"-I{INCLUDE}", f"-I{CSRC}",
]


# Host C: -ffp-contract=off keeps the RoPE frequency expression in plain fp32 steps.
CFLAGS = [
    "-O2", "-std=gnu11", "-fPIC", "-fvisibility=hidden", "-ffp-contract=off", "-Wall", "-Wextra",
    "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include", f"-I{INCLUDE}", f"-I{CSRC}",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm required to build libtkm_attn.so)")


def _compile(src: str, obj: str, extra) -> None:
    if src.endswith(".c"):
        cmd = [os.environ.get("CC", "gcc"), *CFLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    else:
        cmd = [hipcc(), *HIPFLAGS, *extra, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed for {src}:\n{r.stdout}\n{r.stderr}")
    if r.stderr.strip() and src.endswith(".c"):
        raise RuntimeError(f"warnings in {src} (host C builds warning-free):\n{r.stderr}")


def llvm_tool(name: str) -> str:
    for cand in (os.path.join(ROCM, "llvm", "bin", name), os.path.join(ROCM, "lib", "llvm", "bin", name)):
        if os.path.exists(cand):
            return cand
    raise RuntimeError(f"{name} not found under {ROCM}")


def _run(cmd, what):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")


def build_asm_kernel(module: str, symbol: str, objdir: str) -> str:
    """Generate, assemble and link one assembly kernel; returns the object file of a C
    translation unit that holds its code object as `<symbol>_co` / `<symbol>_co_size`."""
    import importlib
    gen = importlib.import_module(module)
    s_path = os.path.join(objdir, symbol + ".s")
    dt = symbol.rsplit("_", 1)[1]          # the element type ends the symbol: _f16, _bf16
    with open(s_path, "w") as f:
        f.write(gen.build() if dt == "f16" else gen.build(dt=dt))
    o_path = os.path.join(objdir, symbol + ".o")
    co_path = os.path.join(objdir, symbol + ".co")
    _run([llvm_tool("clang"), "-x", "assembler", "-target", "amdgcn-amd-amdhsa", f"-mcpu={ARCH}",
          "-c", s_path, "-o", o_path], f"assembling {symbol}")
    _run([llvm_tool("ld.lld"), "-shared", o_path, "-o", co_path], f"linking {symbol}")
    with open(co_path, "rb") as f:
        blob = f.read()
    c_path = os.path.join(objdir, symbol + "_co.c")
    with open(c_path, "w") as f:
        f.write(f"/* code object of {symbol} (generated by {module}) */\n")
        f.write(f"const unsigned long {symbol}_co_size = {len(blob)}ul;\n")
        f.write(f"__attribute__((aligned(4096))) const unsigned char {symbol}_co[] = {{\n")
        for i in range(0, len(blob), 24):
            f.write(",".join(str(b) for b in blob[i:i + 24]) + ",\n")
        f.write("};\n")
    obj = os.path.join(objdir, symbol + "_co.o")
    _run([os.environ.get("CC", "gcc"), "-O1", "-fPIC", "-c", c_path, "-o", obj], f"compiling {symbol} blob")
    return obj


def build(verbose: bool = False, extra=()) -> str:
    objdir = os.path.join(PKG, "_obj")
    os.makedirs(objdir, exist_ok=True)
    if ROOT not in sys.path:
        sys.path.insert(0, ROOT)
    srcs = SOURCES + C_SOURCES + RT_SOURCES + RT_C_SOURCES
    objs = [os.path.join(objdir, s.replace(".", "_") + ".o") for s in srcs]
    with ThreadPoolExecutor(max_workers=min(len(srcs), 8)) as ex:
        list(ex.map(lambda so: _compile(so[0], so[1], extra), zip(srcs, objs)))
    asm_objs = [build_asm_kernel(m, sym, objdir) for m, sym in ASM_KERNELS]
    n_attn = len(SOURCES) + len(C_SOURCES)
    _link(objs[:n_attn] + asm_objs, LIB_PATH, ["-lhiprtc"])
    _link(objs + asm_objs, HIP_LIB_PATH, ["-lhiprtc", "-lhipblaslt"])
    if verbose:
        print(f"built {LIB_PATH} and {HIP_LIB_PATH}")
    return LIB_PATH


def _link(objs, out, libs) -> None:
    tmp = out + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp, f"-L{ROCM}/lib", *libs,
           f"-Wl,-rpath,{ROCM}/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, out)


if __name__ == "__main__":
    build(verbose=True, extra=sys.argv[1:])
