"""Builds ``libmi355_ops.so`` (the C-ABI library) from the HIP sources in ``csrc/`` for gfx950."""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libmi355_ops.so")

SOURCES = ["context.hip", "dw_reduce.hip", "norm.hip", "eltwise.hip", "qknorm_rope.hip", "embed.hip", "softmax_ce.hip", "optim.hip",
           "staging.hip", "bf16_ops.hip", "gemm.hip", "ckpt.hip", "host_dropins.hip"]

# -ffp-contract=off: products and sums round separately, as the reference's sequences of vDSP calls do;
# the packed-fp32 feature is disabled because some packed forms have given wrong results on this hardware.
# -amdgpu-kernarg-preload-count: the dispatcher puts the first 14 dwords of a kernel's arguments into the registers of its waves,
# which otherwise begin with a trip to memory for them before they can ask for anything else: 0.1 to 0.2 us of every launch
# (the five launches of the fp16 / INT8 hand-over 58.8 -> 57.9 us, an odd layer's ten 70.6 -> 69.4, a bfloat16 loss of
# [32000][200], one launch, 14.9 -> 14.7).
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-ffp-contract=off",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wall", "-Wno-unused-function",
         "-Wno-unknown-attributes", "-mllvm", "-amdgpu-kernarg-preload-count=16"]


def _hipcc():
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if c and (os.path.isabs(c) and os.path.exists(c) or not os.path.isabs(c)):
            return c
    return "hipcc"


def build(verbose=False, jobs=7):
    """Compile every source (always recompiles) and link the shared library. Returns its path."""
    os.makedirs(OBJ, exist_ok=True)
    hipcc = _hipcc()

    def compile_one(src):
        obj = os.path.join(OBJ, src.replace(".hip", ".o"))
        cmd = [hipcc] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0 or verbose:
            sys.stderr.write(r.stdout + r.stderr)
        if r.returncode != 0:
            raise RuntimeError("hipcc failed on %s" % src)
        return obj

    with ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(compile_one, SOURCES))
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs + ["-ldl"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("link failed")
    return LIB


HOST_SRC = os.path.join(HERE, "host", "train_step_mirror.c")
HOST_BIN = os.path.join(HERE, "host", "train_step_mirror")


def build_host_mirror():
    """Compile the C mirror of the reference's training-step op sequence against the library (gcc)."""
    inc = os.path.join(os.path.dirname(HERE), "include")
    cmd = ["gcc", "-O2", "-std=c99", "-ffp-contract=off", "-Wall", "-I", inc, HOST_SRC, "-L", HERE, "-lmi355_ops",
           "-Wl,-rpath,$ORIGIN/..", "-lm", "-o", HOST_BIN]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("gcc failed on train_step_mirror.c")
    return HOST_BIN


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
    print(build_host_mirror())
