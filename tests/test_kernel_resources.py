"""What the compiler gave the solver kernels whose speed depends on values staying in registers: scratch
memory per lane and LDS, from the metadata of the built library's gfx950 code."""

import os
import re
import shutil
import struct
import subprocess

import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "box2d_amd", "lib", "libbox2d_amd.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Kernel name -> (scratch bytes per lane, LDS bytes)."""
    if not os.path.exists(LIB) or not os.path.exists(READELF):
        pytest.skip("needs the built library and llvm-readelf")
    with open(LIB, "rb") as f:
        raw = f.read()
    out = {}
    path = str(tmp_path_factory.mktemp("code") / "object")
    for m in re.finditer(MAGIC, raw):
        at = m.start() + len(MAGIC)
        (entries,) = struct.unpack_from("<Q", raw, at)
        at += 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", raw, at)
            triple = raw[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" not in triple:
                continue
            with open(path, "wb") as f:
                f.write(raw[m.start() + offset:m.start() + offset + size])
            notes = subprocess.run([READELF, "--notes", path], capture_output=True, text=True, check=True).stdout
            for kernel in re.split(r"\n  - ", notes):
                field = {k: re.search(rf"\.{k}:\s+(\S+)", kernel) for k in ("symbol", "private_segment_fixed_size",
                                                                             "group_segment_fixed_size")}
                if all(field.values()):
                    out[field["symbol"][1]] = (int(field["private_segment_fixed_size"][1]),
                                               int(field["group_segment_fixed_size"][1]))
    return out


# The XCD solver's forms for worlds with joints: a joint's two bodies are in its lane's registers.
@pytest.mark.parametrize("name,scratch", [("SolveFlowKernelILi4ELi256ELb1E", 0), ("SolveFlowKernelILi2ELi512ELb1E", 64),
                                          ("SolveFlowKernelILi4ELi256ELb0E", 0), ("SolveFlowKernelILi2ELi512ELb0E", 64)])
def test_xcd_solver(kernels, name, scratch):
    found = [v for k, v in kernels.items() if name in k]
    assert len(found) == 1
    assert found[0][0] <= scratch and found[0][1] <= 64, found


@pytest.mark.parametrize("threads", [512, 1024])
def test_batch_solver_without_general_worlds(kernels, threads):
    found = [v for k, v in kernels.items() if f"SolveFusedBatchKernelILi{threads}ELb0E" in k]
    assert len(found) == 1 and found[0][0] == 0, found
