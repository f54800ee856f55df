"""The copies from global memory into LDS, in the code the compiler made.

A load into LDS takes its LDS base from M0, and after a scalar write of M0
the hardware needs one wait state (any instruction) before such a load.  The
compiler keeps it for the instructions it emits; inside inline asm nobody
does but the source.
"""
from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from nanokv import build as nkv_build


def instructions(library: Path, folder: Path):
    """(kernel, instruction text) of the gfx950 code objects of the built library."""
    objdump = Path(nkv_build.hipcc_path()).resolve().parents[1] / "llvm" / "bin" / "llvm-objdump"
    if not objdump.is_file():
        pytest.skip(f"no {objdump}")
    copy = folder / "library.so"
    shutil.copy(library, copy)
    subprocess.run([objdump, "--offloading", copy.name], cwd=folder, check=True, capture_output=True)
    for code in sorted(folder.glob(f"*{nkv_build.OFFLOAD_ARCH}")):
        listing = subprocess.run([objdump, "-d", "--no-show-raw-insn", code.name], cwd=folder,
                                 check=True, capture_output=True, text=True).stdout
        kernel = ""
        for line in listing.splitlines():
            label = re.match(r"[0-9a-f]+ <(.*)>:$", line)
            if label:
                kernel = label[1]
            elif line.startswith("\t"):
                yield kernel, line.split("//")[0].strip()


def test_a_wait_state_between_an_m0_write_and_a_load_into_lds(tmp_path):
    assert nkv_build.LIBRARY_PATH.is_file(), "build the library first"
    loads, hazards, before = 0, [], ""
    for kernel, text in instructions(nkv_build.LIBRARY_PATH, tmp_path):
        if re.match(r"(global_load_lds|buffer_load.* lds)", text):
            loads += 1
            if re.match(r"s_\w+ m0,", before):
                hazards.append((kernel, before, text))
        before = text
    assert loads > 0  # the attention kernels copy this way
    assert not hazards, f"{len(hazards)} of {loads} loads, first {hazards[0]}"
