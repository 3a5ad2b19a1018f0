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
# 120 moves beside 40 products of the GEMM's smaller tiles, and the one-item prefill takes
# 4 to 7 % longer at head_dim 64 (1x32x2048x64: 47.4 us against 44.2), the decode over a
# contiguous cache 2 to 3 % (64 sequences of 100 to 3000 tokens, 16 heads of 64: 94.9 us
# against 92.2; 64 x 4096, 8 heads of 128: 89 against 87).
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
