"""The stage kernels of every unit of the built library are call-free: the sources are compiled in several
units, and each unit's kernels come in a bundle of their own inside the library (in link order)."""
import subprocess
from pathlib import Path

import pytest

from pyhype_amd import _native as nat

LLVM = Path("/opt/rocm/llvm/bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.mark.skipif(not (LLVM / "llvm-objdump").exists(), reason="ROCm LLVM tools not available")
def test_no_stage_unit_makes_a_function_call(tmp_path):
    from pyhype_amd._build import SOURCES

    fat = tmp_path / "fat.bin"
    subprocess.run([str(LLVM / "llvm-objcopy"), f"--dump-section=.hip_fatbin={fat}", str(nat.LIB_PATH),
                    str(tmp_path / "host.so")], check=True, capture_output=True)
    data = fat.read_bytes()
    starts = [i for i in range(0, len(data), 8) if data.startswith(MAGIC, i)]
    assert len(starts) == len(SOURCES)
    kernels = 0
    for n, (a, b) in enumerate(zip(starts, starts[1:] + [len(data)])):
        one, code = tmp_path / f"{n}.bin", tmp_path / f"{n}.o"
        one.write_bytes(data[a:b])
        subprocess.run([str(LLVM / "clang-offload-bundler"), "--unbundle", "--type=o",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--input={one}", f"--output={code}"], check=True,
                       capture_output=True)
        dis = subprocess.run([str(LLVM / "llvm-objdump"), "-d", "--mcpu=gfx950", str(code)], check=True,
                             capture_output=True, text=True).stdout
        if SOURCES[n] == "phx_adjoint.hip":
            continue
        kernels += dis.count("s_endpgm")
        assert "s_swappc" not in dis, SOURCES[n]
    assert kernels > 100
