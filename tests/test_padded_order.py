"""Which sequence the workgroups of a padded forward take whose sequences lie side by side (padded_sequence, device_common.h),
on the CPU: every row of every sequence once, and no sequence on a few of the 32 queues alone to which the hardware deals workgroups
by their linear id."""
from __future__ import annotations

import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

from test_kernel_resources import CSRC, HIPCC

pytestmark = pytest.mark.skipif(shutil.which(HIPCC) is None, reason="hipcc not installed")
SOURCE = """
#include "device_common.h"
extern "C" void order(int heads, int batch, int items, int32_t *sequence) {
  const int shift = dk::padded_shift(heads, batch);
  for (int z = 0; z < items; ++z)
    for (int y = 0; y < batch; ++y) sequence[z * batch + y] = dk::padded_sequence(y, z, batch, shift);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = str(tmp_path_factory.mktemp("order"))
    with open(os.path.join(d, "order.hip"), "w") as f:
        f.write(SOURCE)
    subprocess.run([HIPCC, "--cuda-host-only", "-x", "hip", "-O1", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, os.path.join(d, "order.hip"),
                    "-o", os.path.join(d, "order.so")], check=True, capture_output=True)
    return C.CDLL(os.path.join(d, "order.so"))


@pytest.mark.parametrize("heads", [1, 2, 3, 4, 6, 8, 12, 16, 24, 28, 32, 40])
@pytest.mark.parametrize("batch", [2, 3, 4, 5, 6, 7, 8, 12, 16])
def test_every_sequence_goes_round_all_queues(lib, heads, batch):
    items = 32 * batch
    out = (C.c_int32 * (items * batch))()
    lib.order(heads, batch, items, out)
    sequence = np.array(out).reshape(items, batch)
    assert (np.sort(sequence, axis=1) == np.arange(batch)).all()
    z, y, x = np.meshgrid(np.arange(items), np.arange(batch), np.arange(heads), indexing="ij")
    queue = (x + heads * (y + batch * z)) % 32
    for b in range(batch):
        mine = np.bincount(queue[sequence[z, y] == b], minlength=32)
        assert mine.max() <= 2.01 * mine.mean(), (b, mine)
