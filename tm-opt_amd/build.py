"""In-tree build of libtmopt_attn.so for gfx950.

The HIP sources of csrc/ are compiled side by side (one hipcc each) and
linked into lib/libtmopt_attn.so. Packed FP32 instructions are disabled for all device
code (-packed-fp32-ops); the host pass warns that it does not know the
feature, which is harmless.
"""
import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIB_DIR, "libtmopt_attn.so")
ARCH = os.environ.get("TMOPT_ARCH", "gfx950")

SOURCES = ["capi.hip", "kv_write.hip", "decode.hip", "prefill.hip",
           "prefill_split.hip"]

FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def hipcc():
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    cand = os.path.join(rocm, "bin", "hipcc")
    return cand if os.path.exists(cand) else "hipcc"


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        sys.stderr.write(err + "\n")
        raise subprocess.CalledProcessError(res.returncode, cmd, res.stdout,
                                            err)
    if verbose and err.strip():
        sys.stderr.write(err + "\n")


def build(verbose=False):
    """Compile every source; raise CalledProcessError on failure."""
    os.makedirs(LIB_DIR, exist_ok=True)
    tmp = LIB + ".tmp"
    with tempfile.TemporaryDirectory() as d:
        objs = [os.path.join(d, os.path.splitext(s)[0] + ".o")
                for s in SOURCES]
        cmds = [[hipcc()] + FLAGS + ["-c", os.path.join(CSRC, s), "-o", o]
                for s, o in zip(SOURCES, objs)]
        with ThreadPoolExecutor(len(cmds)) as pool:
            list(pool.map(lambda c: _run(c, verbose), cmds))
        _run([hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC"] + objs +
             ["-o", tmp], verbose)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
