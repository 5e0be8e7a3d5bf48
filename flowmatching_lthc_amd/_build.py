"""Build liblthc_hip.so (gfx950) in-tree with hipcc.

Usage: ``python -m flowmatching_lthc_amd._build``.  The library lands in
``flowmatching_lthc_amd/_lib/`` where ``_abi.py`` loads it; nothing is
compiled at import time.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
SOURCES = [os.path.join(PKG, "csrc", n) for n in ("lthc_kernels.hip", "branch.hip")]
LIB_DIR = os.path.join(PKG, "_lib")
LIB_PATH = os.path.join(LIB_DIR, "liblthc_hip.so")
ARCH = "gfx950"

# -packed-fp32-ops keeps the compiler from forming v_pk_{add,mul,fma}_f32.
HIPCC_FLAGS = [
    "-O3",
    "-std=c++17",
    f"--offload-arch={ARCH}",
    "-fPIC",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-I",
    os.path.join(ROOT, "include"),
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found (ROCm toolchain required to build liblthc_hip.so)")
    return path


def build(verbose: bool = False) -> str:
    """Compile every HIP source (side by side) and link them into LIB_PATH; returns the path."""
    os.makedirs(LIB_DIR, exist_ok=True)
    tmp = LIB_PATH + ".tmp"
    with tempfile.TemporaryDirectory(dir=LIB_DIR) as work:
        objects = [os.path.join(work, os.path.basename(src) + ".o") for src in SOURCES]
        cmds = [[hipcc(), *HIPCC_FLAGS, "-c", "-o", obj, src] for src, obj in zip(SOURCES, objects)]
        procs = [subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True) for cmd in cmds]
        outputs = [p.communicate()[0] for p in procs]
        link = [hipcc(), f"--offload-arch={ARCH}", "-fPIC", "-shared", "-o", tmp, *objects]
        for cmd, p, text in zip(cmds, procs, outputs):
            if p.returncode != 0:
                raise RuntimeError(f"hipcc failed ({p.returncode}):\n{' '.join(cmd)}\n{text[-4000:]}")
            if verbose and text.strip():
                print(text, file=sys.stderr)
        proc = subprocess.run(link, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"hipcc failed ({proc.returncode}):\n{' '.join(link)}\n{proc.stderr[-4000:]}")
    os.replace(tmp, LIB_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
