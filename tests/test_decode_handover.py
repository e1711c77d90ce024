"""Build-time check of the decode kernels' hand-over between workgroups (no GPU needed): the workgroup
that arrives last at a row reads partials that workgroups on other dies have written, so the arrival
- the one 64-bit atomic addition of these kernels - has to release this workgroup's stores (write back
its die's L2, then wait) and acquire the others' (invalidate) before the barrier that lets the
workgroup's other waves read."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from test_kernel_resources import CSRC, FLAGS, HIPCC, _extra_flags


@pytest.mark.skipif(shutil.which(HIPCC) is None, reason="hipcc not installed")
def test_arrival_releases_and_acquires_at_device_scope(tmp_path):
    asm = str(tmp_path / "decode.s")
    flags = [f for f in FLAGS if not f.startswith("-Rpass") and f != "-c"]
    subprocess.run([HIPCC, *flags, *_extra_flags("decode.hip"), "-S", os.path.join(CSRC, "decode.hip"), "-o", asm],
                   check=True, capture_output=True)
    with open(asm) as f:
        kernels = re.findall(r"^(_ZN2dk21decode_partial_kernel\S*):(.*?)^\.Lfunc_end", f.read(), re.M | re.S)
    assert len(kernels) > 10
    for name, body in kernels:
        code = [x.split(";")[0].strip() for x in body.splitlines()]
        code = [x for x in code if x and not x.startswith(".")]
        adds = [i for i, x in enumerate(code) if x.startswith("global_atomic_add_x2")]
        assert len(adds) == 1, name
        at = adds[0]
        # everything between the write-back and the addition: the wait for it
        back = max(i for i, x in enumerate(code[:at]) if x.startswith("buffer_wbl2"))
        assert code[back] == "buffer_wbl2 sc1" and any("vmcnt(0)" in x for x in code[back + 1:at]), name
        # every wave's stores have arrived ahead of the barrier in front of the addition
        barrier = max(i for i, x in enumerate(code[:back]) if x == "s_barrier")
        assert any("vmcnt(0)" in x for x in code[max(0, barrier - 8):barrier]), name
        behind = next(i for i in range(at, len(code)) if code[i] == "s_barrier")
        assert "buffer_inv sc1" in code[at + 1:behind], name
