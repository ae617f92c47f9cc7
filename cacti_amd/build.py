"""Builds libcacti_gpu_hip_ffi.so for gfx950 with hipcc (cross-compiles without a GPU).

    python -m cacti_amd.build            # compile every source and link
"""
import os
import shutil
import subprocess
import sys
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor

from cacti_amd import asm_check

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "lib")
LIB = os.path.join(OUT_DIR, "libcacti_gpu_hip_ffi.so")
FAST = os.path.join(OUT_DIR, "_fast.so")       # CPython functions over LIB (pysrc/fast.cpp)

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-fvisibility=hidden",
    "-ffp-contract=off",                       # keep the reference's per-thunk rounding points
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-value", "-Wno-unused-result", "-Wno-unknown-warning-option",
]
# Sources with matrix instructions or loads into LDS in inline assembly: what the compiler made of them is checked.  In
# gemm_direct.hip, whose kernels hold all of a wave's registers, a spill and a product rounded only once are faults too.
CHECKED = ("attention.hip", "attention_short.hip", "gemm_direct.hip", "gemm_mfma.hip")
# kernels of which a CU is to hold four workgroups: the products of many tiles and operands of any alignment
REGISTERS = {"gemm_direct.hip": [(r"gemm_part_kernel.*Lb1EEEv", 128)]}


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp")))


def _compile(src):
    name = os.path.splitext(src)[0]
    obj = os.path.join(OUT_DIR, name + ".o")
    if src not in CHECKED:
        _hipcc(src, obj)
        return obj
    with tempfile.TemporaryDirectory() as tmp:
        made = os.path.join(tmp, name + ".o")
        _hipcc(src, made, "--save-temps=obj")
        asm = [f for f in os.listdir(tmp) if f.endswith("gfx950.s")]
        if len(asm) != 1:
            raise RuntimeError("%s: no assembly to check among %s" % (src, sorted(os.listdir(tmp))))
        with open(os.path.join(tmp, asm[0])) as f:
            faults = asm_check.check(f.read(), spills=src == "gemm_direct.hip", fused=src == "gemm_direct.hip",
                                     registers=REGISTERS.get(src, ()))
        if faults:
            raise RuntimeError("%s: %d faults around inline assembly\n%s" % (src, len(faults), "\n".join(faults[:20])))
        shutil.move(made, obj)
    return obj


def _hipcc(src, obj, *more):
    cmd = [HIPCC] + FLAGS + (["-x", "hip"] if src.endswith(".cpp") else []) + \
          ["-c", os.path.join(CSRC, src), "-o", obj] + list(more)
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in p.stdout.splitlines()
                    if "is not a recognized feature for this target" not in l)
    if p.returncode != 0:
        raise RuntimeError("hipcc failed on %s:\n%s" % (src, out))
    if out.strip():
        sys.stderr.write(out + "\n")


def build(jobs=4):
    os.makedirs(OUT_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, sources()))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
    subprocess.check_call(cmd)
    import torch
    from torch.utils import cpp_extension
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    subprocess.check_call(
        ["g++", "-O2", "-shared", "-fPIC", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
         "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI, "-I" + sysconfig.get_paths()["include"]] +
        [f for d in cpp_extension.include_paths() + [os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include")]
         for f in ("-isystem", d)] +
        [os.path.join(HERE, "pysrc", "fast.cpp"), "-o", FAST, "-L" + OUT_DIR, "-l:" + os.path.basename(LIB), "-L" + torch_lib,
         "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python", "-Wl,-rpath,$ORIGIN"])
    return LIB


def ensure():
    """The library's path, built first if no built library is there (tests, the smoke run and the
    benchmark call this; the loader itself never builds and never falls back)."""
    return LIB if os.path.exists(LIB) and os.path.exists(FAST) else build()


if __name__ == "__main__":
    print(build())
