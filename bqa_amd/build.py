"""Build ``bqa_amd/libbqa_hip.so`` in-tree with hipcc for gfx950.

    python -m bqa_amd.build

Every HIP source is compiled with packed FP32 instructions disabled
(``-Xclang -target-feature -Xclang -packed-fp32-ops``).
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
SOURCES = ("bqa_api.hip", "node_gemm.hip", "canon_wide.hip")
OUT = os.path.join(HERE, "libbqa_hip.so")
ARCH = os.environ.get("BQA_OFFLOAD_ARCH", "gfx950")


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def build(verbose: bool = True) -> str:
    flags = [f"--offload-arch={ARCH}", "-O3", "-std=c++20", "-fPIC",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument"]

    def run(cmd):
        if verbose:
            print(" ".join(cmd), flush=True)
        proc = subprocess.run(cmd, capture_output=True, text=True)
        errs = "\n".join(l for l in proc.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
        if proc.returncode != 0:
            raise RuntimeError(f"hipcc failed ({proc.returncode}):\n{errs}")
        if errs and verbose:
            print(errs, file=sys.stderr)

    # the sources hold separate kernels: compiled side by side, then linked
    with tempfile.TemporaryDirectory() as work, ThreadPoolExecutor(len(SOURCES)) as pool:
        objs = [os.path.join(work, f"{name}.o") for name in SOURCES]
        list(pool.map(run, [[hipcc(), *flags, "-c", os.path.join(CSRC, name), "-o", obj]
                            for name, obj in zip(SOURCES, objs)]))
        tmp = OUT + ".tmp"
        run([hipcc(), *flags, "-shared", "-o", tmp, *objs])
    os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build())
