"""Scalar registers of the dQ kernels in the built library (no GPU needed): a launch that cuts no row must not pay for the
code that does.  Folded into one instantiation that code spilled fifty scalars, ten without it, and took launches that
cut nothing 4 - 8 % longer."""
from __future__ import annotations

import os
import re
import shutil
import struct
import subprocess

import pytest

from dkernel_amd import _lib

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def _kernels(tmp):
    """name -> spilled scalars of the kernels in the library's device code"""
    with open(_lib.LIB_PATH, "rb") as f:
        data = f.read()
    found = {}
    for m in re.finditer(b"\x7fELF\x02", data):
        at = m.start()
        if struct.unpack_from("<H", data, at + 18)[0] != 224:  # EM_AMDGPU
            continue
        sections, entry, count = struct.unpack_from("<Q", data, at + 40)[0], *struct.unpack_from("<HH", data, at + 58)
        path = os.path.join(tmp, "code.elf")
        with open(path, "wb") as f:
            f.write(data[at:at + sections + entry * count])
        notes = subprocess.run([READELF, "-n", path], capture_output=True, text=True, check=True).stdout
        for kernel in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel)
            spills = re.search(r"\.sgpr_spill_count:\s+(\d+)", kernel)
            if name and spills:
                found[name.group(1)] = int(spills.group(1))
    return found


@pytest.mark.skipif(shutil.which(READELF) is None, reason="llvm-readelf not installed")
def test_launches_that_cut_nothing_spill_few_scalars(tmp_path):
    kernels = {k: v for k, v in _kernels(str(tmp_path)).items() if "mfma_dq_pair_kernel" in k}
    # <type, tile width, PAD, SUB, CUT, head dims>
    uncut = {k: v for k, v in kernels.items() if re.search(r"Lb[01]ELb[01]ELb0ELi\d+EEEv", k)}
    assert len(kernels) == 40 and len(uncut) == 20, list(kernels)
    assert max(uncut.values()) <= 22, uncut


@pytest.mark.skipif(shutil.which(READELF) is None, reason="llvm-readelf not installed")
def test_fp32_launches_that_cut_nothing_spill_few_scalars(tmp_path):
    kernels = {k: v for k, v in _kernels(str(tmp_path)).items() if "f329dq_kernel" in k}
    uncut = {k: v for k, v in kernels.items() if re.search(r"Lb[01]ELb0EEEv", k)}  # <head dims, PAD, CUT>
    assert len(kernels) == 10 and len(uncut) == 5, list(kernels)
    assert max(uncut.values()) <= 8, uncut
