"""Builds reef_amd/libreef_hip.so: every HIP kernel and the C ABI, for gfx950 only.

Run ``python -m reef_amd._build``; ``__graft_entry__.build()`` calls build().
"""
from __future__ import annotations

import os
import shlex
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
SOURCES = ["quant.hip", "prefill.hip", "prefill_packed.hip", "prefill_cache.hip", "decode.hip",
           "kv_append.hip", "int_head.hip", "linear.hip"]
LIB = os.path.join(PKG, "libreef_hip.so")

FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # No packed fp32 instructions (v_pk_{add,mul,fma}_f32) in device code.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-result",
    "-I", os.path.join(ROOT, "include"),
]


# Per source: matrix products with their accumulators in ordinary vector registers. Left to
# itself the compiler moves accumulators between the two register files inside the loops:
# 120 moves beside 40 products of the GEMM's smaller tiles (256 x 8192 -> 8192: 41 us with its
# row quantization, 33.6 this way; 300 x 2048 -> 2048 13.4 against 12.9), the balanced prefill
# with per-token scales takes 3 to 6 % longer (1x16x1024x128: 40.8 us against 38.5), the
# decode over a contiguous cache 0.4 % (64 x 4096, 8 heads of 128: 89.6 us against 89.3). The
# other kernels of prefill.hip and those of int_head.hip come out the same either way.
VGPR_FORM = ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]
SOURCE_FLAGS = {s: VGPR_FORM for s in ("linear.hip", "prefill.hip", "decode.hip")}


def commands(objdir):
    """One compile command per source, then the link command."""
    objs = [os.path.join(objdir, s.replace(".hip", ".o")) for s in SOURCES]
    compiles = [["hipcc", *FLAGS, *SOURCE_FLAGS.get(s, []), "-c", os.path.join(PKG, "csrc", s),
                 "-o", o] for s, o in zip(SOURCES, objs)]
    return compiles, ["hipcc", "--offload-arch=gfx950", "-fPIC", "-shared", "-o", LIB + ".tmp",
                      *objs]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(shlex.quote(c) for c in cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # The host pass does not know the packed-fp32 feature name; that warning is noise.
    noise = "is not a recognized feature for this target"
    msgs = [l for l in (proc.stdout + proc.stderr).splitlines() if noise not in l]
    if proc.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + "\n".join(msgs))
    if msgs and verbose:
        print("\n".join(msgs))


def build(verbose: bool = False) -> str:
    with tempfile.TemporaryDirectory() as objdir:
        compiles, link = commands(objdir)
        with ThreadPoolExecutor(min(4, len(compiles))) as pool:
            list(pool.map(lambda c: _run(c, verbose), compiles))
        _run(link, verbose)
    os.replace(LIB + ".tmp", LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
