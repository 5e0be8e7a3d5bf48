"""Build liblthc_hip.so (gfx950, hipcc) and lthc_torch.so (the native torch operators on it, g++) in-tree.

Usage: ``python -m flowmatching_lthc_amd._build``.  The libraries land in
``flowmatching_lthc_amd/_lib/`` where ``_abi.py`` loads them; nothing is
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
OPS_SOURCE = os.path.join(PKG, "csrc", "torch_ops.cpp")
OPS_PATH = os.path.join(LIB_DIR, "lthc_torch.so")
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


def cxx() -> str:
    path = shutil.which("g++")
    if path is None:
        raise RuntimeError("g++ not found (needed to build lthc_torch.so)")
    return path


def _torch_flags() -> tuple[list[str], list[str]]:
    """(compile, link) flags of a host-only torch extension on ROCm."""
    import torch  # imported here: only the build needs torch's headers

    root = os.path.dirname(torch.__file__)
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    compile_flags = [
        "-O2", "-std=c++17", "-fPIC", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
        "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-isystem", os.path.join(root, "include"),
        "-isystem", os.path.join(root, "include", "torch", "csrc", "api", "include"),
        "-isystem", os.path.join(rocm, "include"),
    ]  # fmt: skip
    # torch's own libraries are loaded before this one; liblthc_hip.so lies beside it
    link_flags = [
        "-shared", "-L", LIB_DIR, "-llthc_hip", "-Wl,-rpath,$ORIGIN", "-L", os.path.join(root, "lib"),
        "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch",
    ]  # fmt: skip
    return compile_flags, link_flags


def build(verbose: bool = False) -> str:
    """Compile every source (side by side) and link LIB_PATH and OPS_PATH; returns LIB_PATH."""
    os.makedirs(LIB_DIR, exist_ok=True)

    def check(cmd: list[str], rc: int, text: str) -> None:
        if rc != 0:
            raise RuntimeError(f"{os.path.basename(cmd[0])} failed ({rc}):\n{' '.join(cmd)}\n{text[-4000:]}")
        if verbose and text.strip():
            print(text, file=sys.stderr)

    def link(cmd: list[str], out: str) -> None:
        proc = subprocess.run([*cmd, "-o", out + ".tmp"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
        check(cmd, proc.returncode, proc.stdout)
        os.replace(out + ".tmp", out)

    torch_compile, torch_link = _torch_flags()
    with tempfile.TemporaryDirectory(dir=LIB_DIR) as work:
        objects = [os.path.join(work, os.path.basename(src) + ".o") for src in SOURCES]
        ops_object = os.path.join(work, "torch_ops.o")
        cmds = [[hipcc(), *HIPCC_FLAGS, "-c", "-o", obj, src] for src, obj in zip(SOURCES, objects)]
        cmds.append([cxx(), *torch_compile, "-c", "-o", ops_object, OPS_SOURCE])
        procs = [subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True) for cmd in cmds]
        outputs = [p.communicate()[0] for p in procs]
        for cmd, p, text in zip(cmds, procs, outputs):
            check(cmd, p.returncode, text)
        link([hipcc(), f"--offload-arch={ARCH}", "-fPIC", "-shared", *objects], LIB_PATH)
        link([cxx(), ops_object, *torch_link], OPS_PATH)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
