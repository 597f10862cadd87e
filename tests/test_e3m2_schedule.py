"""How the E3M2 GEMM's main tile orders its operands: csrc/gemm_e3m2_tile.h compiled for the CPU
with stand-ins for its loads, waits and barriers (tests/host/e3m2_tile), at every tile height,
plain and GELU, short k ranges and walks over several tiles.  A row operand that a wave's own
counted waits and the barriers do not cover is an error there, while on the GPU it only shows
when a load happens to be late."""

from __future__ import annotations

import importlib.util
import os
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "pi05-pytorch-fast_amd" / "csrc"


def _emulate(tmp_path: Path, *flags: str) -> subprocess.CompletedProcess:
    for f in (ROOT / "tests" / "host" / "e3m2_tile").iterdir():
        shutil.copy(f, tmp_path)
    shutil.copy(CSRC / "gemm_e3m2_tile.h", tmp_path)  # beside the stand-ins, which its includes then find
    rocm = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
    exe = tmp_path / "emulate"
    subprocess.run([str(rocm / "llvm" / "bin" / "clang++"), "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    f"-I{rocm / 'include'}", f"-I{CSRC}", *flags, str(tmp_path / "emulate.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)


def test_every_row_operand_is_covered_by_the_counted_waits(tmp_path):
    run = _emulate(tmp_path)
    assert run.returncode == 0, run.stdout[-3000:]


@pytest.mark.parametrize("loose", [1, 3])
def test_the_emulation_notices_a_count_that_is_too_large(tmp_path, loose):
    run = _emulate(tmp_path, f"-DEMULATE_LOOSE={loose}")
    for mi in (4, 5, 6, 7):
        for form in ("plain", "GELU"):
            assert f"MI {mi} {form}, 16 k blocks" in run.stdout


@pytest.mark.parametrize("unit,kernels,count", [
    ("gemm.hip", r"gemm_w4a4_kernelILi[4-7]ELi4ELi4ELi1ELb[01]ELi2ELi2ELb0ELb0ELb1E", 8),
    ("quant_rot.hip", r"fwht_quant_kernelILi14E", 3)])
def test_no_register_spills(tmp_path, unit, kernels, count):
    """The main tile's kernels keep everything in registers (a spilled value's reload waits for all
    the loads that the rings hold in flight), and so do the K = 16384 quantizers."""
    spec = importlib.util.spec_from_file_location("_build_lib", CSRC.parent / "build_lib.py")
    build_lib = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build_lib)
    cmds, _ = build_lib.compile_commands(["gfx950"], tmp_path)
    cmd = next(c for c in cmds if c[c.index("-c") + 1].endswith(unit))
    asm = tmp_path / "unit.s"
    cmd = [a for a in cmd if a != "-c"]
    cmd[cmd.index("-o") + 1] = str(asm)
    subprocess.run(cmd + ["-S", "--cuda-device-only"], check=True, capture_output=True)
    scratch = re.findall(r"\.set (\S*)\.private_seg_size, (\d+)", asm.read_text())
    found = {n: int(v) for n, v in scratch if re.search(kernels, n)}
    assert len(found) == count and not any(found.values()), found


def test_direct_loads_declare_their_register():
    """m0, which the direct loads' asm writes, is among what it clobbers, and one helper has it."""
    writes = {f.name: f.read_text().count("s_mov_b32 m0") for f in CSRC.iterdir()}
    assert {n: c for n, c in writes.items() if c} == {"direct_load.h": 1}
    assert re.search(r's_mov_b32 m0[^;]*"m0"\)', (CSRC / "direct_load.h").read_text())
