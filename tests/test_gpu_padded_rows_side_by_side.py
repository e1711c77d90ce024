"""Padded prompts: launches of up to 4096 workgroups of at least six rows (pairs of rows) a sequence and three sequences take
the rows of all sequences side by side (for_rows, mfma_fwd.hip).  Every sequence as by itself, the rows of padding cleared."""
from __future__ import annotations

import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, _lib
from helpers import LSE_TOL, TOL, assert_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("heads,kv_heads,dim,block,longest,batch,side_by_side", [
    (8, 8, 64, 64, 500, 9, False),     # row pairs: five and
    (8, 8, 64, 64, 640, 9, True),      # six of them
    (8, 8, 64, 64, 700, 9, True),
    (16, 4, 128, 64, 900, 6, True),    # four heads a workgroup
    (16, 8, 96, 64, 900, 9, True),     # two heads a workgroup, zero-padded tile
    (8, 8, 128, 32, 1500, 8, True),    # masked tiles, row pairs; the sequences move on with every item
    (12, 12, 64, 32, 1100, 7, True),
    (16, 4, 256, 64, 700, 5, True),    # (with every second)
    (16, 16, 128, 64, 2000, 4, True),
    (32, 32, 64, 64, 1900, 2, False),
    (32, 32, 64, 64, 1900, 3, True),
    (32, 32, 64, 64, 1800, 8, True),   # 4096 workgroups
    (32, 32, 64, 64, 1930, 8, False),  # and more
])
@pytest.mark.parametrize("padding", ["left", "right"])
def test_every_sequence_as_by_itself(heads, kv_heads, dim, block, longest, batch, side_by_side, padding):
    lens = [max(1, longest * (i * 5 % batch + 1) // batch) for i in range(batch)]
    lens[1] = 1
    g = torch.Generator(device=DEV).manual_seed(longest)
    q, k, v = (torch.randn(batch, longest, h, dim, generator=g, device=DEV, dtype=torch.bfloat16)
               for h in (heads, kv_heads, kv_heads))
    mod = LocalStrideSparseAttention(heads, longest, block, 256 // block, 4, num_kv_heads=kv_heads).to(DEV)
    n = torch.tensor(lens, dtype=torch.int32, device=DEV)
    lengths = {"left_paddings": longest - n} if padding == "left" else {"seqlens": n}
    out, lse = mod(q, k, v, dim ** -0.5, return_lse=True, **lengths)
    ran = _lib.lib().dk_last_kernels().decode()
    assert ran.startswith("mfma_fwd_kernel, sequences side by side" if side_by_side else "mfma_fwd_kernel "), ran
    for i, l in enumerate(lens):
        rows = slice(longest - l, longest) if padding == "left" else slice(0, l)
        ref, ref_lse = mod(*(x[i:i + 1, rows] for x in (q, k, v)), dim ** -0.5, return_lse=True)
        assert_close("O", out[i:i + 1, rows], ref, **TOL)
        assert_close("LSE", lse[i:i + 1, :, rows], ref_lse, atol=LSE_TOL, rtol=0)
        outside = torch.ones(longest, dtype=torch.bool, device=DEV)
        outside[rows] = False
        assert (out[i, outside] == 0).all()
        assert (lse[i][:, outside] == -float("inf")).all()
