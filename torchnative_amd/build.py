"""Build recipe for libtnhip.so: hipcc for gfx950, in-tree.

Run as ``python -m torchnative_amd.build`` or through ``__graft_entry__.build()``.
"""

from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libtnhip.so")
SOURCES = ["runtime.hip", "qlinear.hip", "qgemm.hip", "qk.hip", "sdpa.hip", "flash64.hip", "flash_any.hip", "decode.hip", "decode_any.hip", "dense.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# -ffp-contract=off: the q4 recurrence and the SDPA softmax are written with the
#   roundings the reference performs; FMAs are spelled out where wanted.
# -fhip-fp32-correctly-rounded-divide-sqrt: Q8_0's d = amax/127 and 1/d must be
#   IEEE divisions (the default, stated explicitly).
# -packed-fp32-ops disabled: no v_pk_*_f32 from the compiler.
# -amdgpu-mfma-vgpr-form: MFMA accumulators in ordinary VGPRs, so the softmax
#   and the rescales read them without v_accvgpr_read/write copies.
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall",
    "-ffp-contract=off", "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-mfma-vgpr-form",
]


def _compile(src: str, verbose: bool) -> str:
    path = os.path.join(CSRC, src)
    obj = os.path.join(CSRC, src.replace(".hip", ".o"))
    cmd = [HIPCC, *FLAGS, "-c", path, "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"hipcc failed on {src}")
    return obj


def build(verbose: bool = False) -> str:
    # one hipcc per source file, side by side (the files are independent)
    jobs = max(1, min(len(SOURCES), int(os.environ.get("MAX_JOBS", os.cpu_count() or 1))))
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = list(pool.map(lambda s: _compile(s, verbose), SOURCES))
    tmp = OUT + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("hipcc link failed")
    os.replace(tmp, OUT)
    for o in objs:
        os.remove(o)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
