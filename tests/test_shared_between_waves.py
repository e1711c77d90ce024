"""Values that every wave of a backward workgroup leaves in LDS and reads back without a barrier (the part of a row or
column that is its own).  That is sound only while each place is stored once and with the same value by all waves: a
place stored twice lets a late wave's first value replace what an earlier wave is about to read.  Read from the source,
without a GPU."""
from __future__ import annotations

import os
import re

import pytest

from test_kernel_resources import CSRC


def _kernels(source):
    """(name, body) of the kernels in a source file; a body ends at the first closing brace in the first column."""
    with open(os.path.join(CSRC, source)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    for m in re.finditer(r"^__global__[^;{]*?(\w+_kernel)\(", text, re.M | re.S):
        yield m.group(1), text[m.end():text.index("\n}", m.end())]


@pytest.mark.parametrize("source,kernels", [("mfma_bwd.hip", {"mfma_dq_pair_kernel", "mfma_dkdv_kernel"}),
                                            ("mfma_f32.hip", {"dkdv_kernel"})])
def test_each_shared_place_is_stored_once(source, kernels):
    seen = set()
    for name, body in _kernels(source):
        if "__shared__ int part[" not in body:
            continue
        seen.add(name)
        places = int(re.search(r"__shared__ int part\[(\d+)\]", body).group(1))
        stored = sorted(int(x) for x in re.findall(r"\bpart\[(\d+)\]\s*=[^=]", body))
        assert stored == list(range(places)), (name, stored)
        assert body.index("part[0] =") < min(m.start() for m in re.finditer(r"readfirstlane\(part\[", body)), name
    assert seen == kernels
