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
DEVICE_FLAGS = ["--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-munsafe-fp-atomics",
                "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                "-Xclang", "-target-feature", "-Xclang", "-fma-mix-insts", "-Wall", "-Wno-unused-function"]
# -structurizecfg-skip-uniform-regions: the update kernels branch on wave-uniform values (how a row is written, the
# precisions of a rating's rows).  By default the compiler structurises those branches as if lanes could disagree: flag
# registers, three branches for a three-way choice, and paths on which no store is issued, so that the waits for row
# loads must assume the fewest stores in between.  Without it a MASCOT rating waits at vmcnt(12..13) instead of (6..7)
# with a dozen scalar instructions fewer.
# -enable-tail-merge=false goes with it: a device-scope store and a cached store of the same registers are one
# instruction until their cache policies are filled in, and merged they become a device-scope store, which for the copies of
# replicated rows serialises at the memory side (an epoch of 250M ratings in 121 ms instead of 28).
# Epochs without -> with the two flags, both libraries in turn on one model (ms; runs of one side differ by 0.1 to 0.5 %):
#                        k = 64: 8M      100M              k = 128: 8M      100M
#   MASCOT, all binary16   5.37 -> 5.19   8.36 -> 8.20        5.81 -> 4.75   11.29 -> 11.08
#   MASCOT, 10 % binary32  6.43 -> 5.94  10.46 -> 9.81        7.58 -> 6.08   15.88 -> 15.71
#   -v 7                   5.27 -> 5.09   8.11 -> 8.00        5.92 -> 4.88   11.85 -> 11.71
#   fp32 SGD               4.52 -> 4.44  12.00 -> 11.98       5.80 -> 5.83   20.25 -> 20.26
#   MPT                    4.61 -> 4.59  12.06 -> 12.08       6.08 -> 6.05   20.15 -> 20.14
#   AFP                    8.42 -> 8.37  13.45 -> 13.40       9.64 -> 9.65   21.72 -> 21.70
#   MuPPET                10.22 -> 10.30 16.97 -> 16.82      11.34 -> 11.32  23.60 -> 23.53
# MASCOT's mixed epochs of 250M ratings are level.  The rows of fp32 SGD, MPT, AFP and MuPPET were taken while their hot-row builds
# stored through row windows; with the branches they have now fp32 SGD at k = 128 gains too (8M 5.26 -> 4.47, 100M 19.90 -> 19.86).
UNIFORM_BRANCH_FLAGS = ["-mllvm", "-structurizecfg-skip-uniform-regions=true", "-mllvm", "-enable-tail-merge=false"]
STRUCTURISED = set()      # files compiled without these flags (none at present; flags are recorded file by file for them)
EXTRA_FLAGS = os.environ.get("MF_HIPCC_FLAGS", "").split()
KERNEL_SOURCES = ["launch_mascot_plain.hip", "launch_mascot_sampled.hip", "launch_mascot_binary16.hip", "launch_muppet.hip", "launch_afp.hip", "hogwild_launch.hip", "launch_sgd_k128.hip",
                  "launch_mem_quant.hip", "aux_kernels.hip", "sort_shuffle.hip", "launch_mascot.hip"]
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
    return DEVICE_FLAGS + ([] if src in STRUCTURISED else UNIFORM_BRANCH_FLAGS) + EXTRA_FLAGS


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
