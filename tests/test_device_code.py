"""The library's device code (no GPU): a device function that is not inlined
must be shorter than a branch reaches (128 KiB).  In a longer one the compiler
makes long branches through s[30:31], which holds the return address, and the
function does not return to its caller."""
import pathlib
import shutil
import subprocess

import pytest

from rocket_amd import build

LLVM = pathlib.Path("/opt/rocm/llvm/bin")
BRANCH_REACH = 4 * 32768  # a signed 16-bit count of dwords


def code_objects(tmp_path):
    lib = tmp_path / "lib.so"
    shutil.copy(build.LIB, lib)
    subprocess.run([LLVM / "llvm-objdump", "--offloading", lib.name], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    return [p for p in tmp_path.iterdir() if "gfx950" in p.name]


def test_functions_return(tmp_path):
    if not (LLVM / "llvm-objdump").exists() or not pathlib.Path(build.LIB).exists():
        pytest.skip("needs the built library and ROCm's llvm-objdump")
    objects = code_objects(tmp_path)
    assert objects
    kernels = 0
    for obj in objects:
        out = subprocess.run([LLVM / "llvm-readelf", "--symbols", "--wide", obj], check=True, capture_output=True,
                             text=True).stdout
        rows = [ln.split() for ln in out.splitlines() if " FUNC " in ln or " OBJECT " in ln]
        described = {r[-1][:-3] for r in rows if r[-1].endswith(".kd")}
        kernels += len(described)
        for r in rows:
            if r[3] == "FUNC" and r[-1] not in described:
                assert int(r[2], 0) < BRANCH_REACH, r[-1]
    assert kernels > 50
