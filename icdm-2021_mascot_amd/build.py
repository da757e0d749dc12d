"""Builds libmascot_hip.so (the gfx950 kernels behind the C ABI of include/mascot_hip.h)
and the quantized_mf / test_mf command lines in-tree with hipcc.  No GPU is needed to build."""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libmascot_hip.so")
CLI = os.path.join(HERE, "quantized_mf")
EVAL = os.path.join(HERE, "test_mf")
FLAGS_RECORD = os.path.join(OBJ, "device_flags.txt")      # what the library beside it was compiled with, a line per translation unit

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
# -ffp-contract=off: every rounding the update rules spell out must happen (fused where the rule calls fma).
# -munsafe-fp-atomics: hardware float atomic adds for the sampled gradient sums.
# packed-fp32-ops disabled: no v_pk_*_f32 code generation.
# fma-mix-insts disabled: v_fma_mix{lo,hi}_f16 rounds fma(a,b,c) once to binary16, but the update rules
# round to binary32 first and then to binary16 (fmaf followed by __float2half); the two differ by one
# binary16 ulp on rare inputs, so the fused form must not be selected.
# -structurizecfg-skip-uniform-regions: the update kernels branch on wave-uniform values (how a row is written, the
# precisions of a rating's rows).  By default the compiler structurises those branches as if lanes could disagree: flag
# registers, three branches for a three-way choice, and paths on which no store is issued, so that the waits for row
# loads must assume the fewest stores in between.  Without it a MASCOT rating waits at vmcnt(12..13) instead of (6..7)
# with a dozen scalar instructions fewer: an epoch of 8M ratings takes 4.74 instead of 5.73 ms, one of 100M 11.13
# instead of 11.31.
# -enable-tail-merge=false goes with it: a device-scope store and a cached store of the same registers are one
# instruction until their cache policies are filled in, and merged they become a device-scope store, which for the copies of
# replicated rows serialises at the memory side.
DEVICE_FLAGS = ["--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-munsafe-fp-atomics",
                "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                "-Xclang", "-target-feature", "-Xclang", "-fma-mix-insts", "-Wall", "-Wno-unused-function",
                "-mllvm", "-structurizecfg-skip-uniform-regions=true", "-mllvm", "-enable-tail-merge=false"] + os.environ.get("MF_HIPCC_FLAGS", "").split()
KERNEL_SOURCES = ["launch_mascot_plain.hip", "launch_mascot_sampled.hip", "launch_mascot_binary16.hip", "launch_muppet.hip", "launch_afp.hip", "hogwild_launch.hip", "launch_mem_quant.hip", "aux_kernels.hip",
                  "sort_shuffle.hip", "launch_mascot.hip"]
HOST_SOURCES = ["train.cpp"]
CLI_SOURCES = ["main.cpp", "io_utils.cpp"]
EVAL_SOURCES = ["test_mf_main.cpp", "io_utils.cpp"]


def _run(cmd):
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in p.stdout.splitlines() if "is not a recognized feature" not in l)
    if p.returncode != 0:
        raise RuntimeError("command failed: %s\n%s" % (" ".join(cmd), out))
    return out


def device_flags(src):
    """The compiler flags of one .hip file."""
    return DEVICE_FLAGS


def flags_record():
    return "".join("%s: %s\n" % (src, " ".join(device_flags(src))) for src in sorted(KERNEL_SOURCES))


def _compile(src):
    obj = os.path.join(OBJ, os.path.splitext(src)[0] + ".o")
    flags = device_flags(src) if src.endswith(".hip") else ["-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include"]
    _run([HIPCC] + flags + ["-c", os.path.join(CSRC, src), "-o", obj])
    return obj


def build(verbose=False):
    os.makedirs(OBJ, exist_ok=True)
    lib_sources = [s for s in KERNEL_SOURCES + HOST_SOURCES if os.path.exists(os.path.join(CSRC, s))]
    with ThreadPoolExecutor(max_workers=8) as ex:
        objs = list(ex.map(_compile, lib_sources))
    if os.path.exists(FLAGS_RECORD):
        os.remove(FLAGS_RECORD)      # none while it may not be the library's
    _run([HIPCC, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", LIB] + objs)
    with open(FLAGS_RECORD, "w") as f:
        f.write(flags_record())
    if all(os.path.exists(os.path.join(CSRC, s)) for s in CLI_SOURCES):
        with ThreadPoolExecutor(max_workers=2) as ex:
            cobjs = list(ex.map(_compile, CLI_SOURCES))
        _run([HIPCC, "-o", CLI] + cobjs + ["-L" + HERE, "-lmascot_hip", "-Wl,-rpath,$ORIGIN"])
    if all(os.path.exists(os.path.join(CSRC, s)) for s in EVAL_SOURCES):
        eobjs = [_compile(s) for s in EVAL_SOURCES]
        _run([HIPCC, "-o", EVAL] + eobjs + ["-L" + HERE, "-lmascot_hip", "-Wl,-rpath,$ORIGIN"])
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
