"""Build of the in-tree HIP library ``pyhype_amd/lib/libpyhype_hip.so`` for gfx950.

The library is compiled with hipcc directly (no JIT cache) so that the built ``.so`` travels with
the source tree.  Floating-point flags: ``-ffp-contract=off`` keeps every multiply and add a
separately rounded IEEE operation, which the bit-for-bit parity with the reference arithmetic
relies on; packed-FP32 instruction selection is disabled.
"""
from __future__ import annotations

import os
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
LIBDIR = PKG / "lib"
LIB = LIBDIR / "libpyhype_hip.so"
INCLUDE = PKG.parent / "include"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-ffp-contract=off",
    "-fno-fast-math",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
]

# the stage kernels' instances are spread over several units: each takes minutes, and they compile in
# parallel
SOURCES = ["phx_stage_yface.hip", "phx_stage_fused.hip", "phx_stage_lin.hip", "phx_stage_recon.hip",
           "phx_stage_shared.hip", "phx_adjoint.hip", "phx_kernels.hip"]


def _run(cmd):
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}): {' '.join(cmd)}\n{res.stdout}\n{res.stderr}")
    return res.stderr


def build_library(verbose: bool = False, extra_flags=None) -> Path:
    """Compile every HIP source into ``lib/libpyhype_hip.so`` (always recompiles)."""
    LIBDIR.mkdir(exist_ok=True)
    tmp = LIB.with_suffix(".so.tmp")
    jobs = max(1, min(len(SOURCES), int(os.environ.get("MAX_JOBS", 0)) or os.cpu_count() or 1, 8))
    with tempfile.TemporaryDirectory(prefix="phx_build_") as tmpdir:
        objs = [str(Path(tmpdir) / s.replace(".hip", ".o")) for s in SOURCES]
        cmds = [[HIPCC, *HIP_FLAGS, *(extra_flags or []), f"-I{INCLUDE}", "-c", str(CSRC / s), "-o", o]
                for s, o in zip(SOURCES, objs)]
        if verbose:
            print("\n".join(" ".join(c) for c in cmds), flush=True)
        with ThreadPoolExecutor(jobs) as pool:
            notes = list(pool.map(_run, cmds))
        if verbose and any(notes):
            print("".join(notes))
        _run([HIPCC, f"--offload-arch={ARCH}", "-fPIC", "-shared", *objs, "-o", str(tmp)])
    os.replace(tmp, LIB)
    return LIB


def build_test_library(verbose: bool = False) -> Path:
    """Compile the tests' native libraries (tests/native/lib{device,inrange,guards}_numerics.so)."""
    native = PKG.parent / "tests" / "native"
    for name in ("device_numerics", "inrange_numerics", "guards_numerics"):
        out = native / f"lib{name}.so"
        tmp = out.with_suffix(".so.tmp")
        cmd = [HIPCC, *HIP_FLAGS, "-shared", f"-I{INCLUDE}", str(native / f"{name}.hip"), "-o", str(tmp)]
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)
        os.replace(tmp, out)
    return out


if __name__ == "__main__":
    print(build_library(verbose=True))
