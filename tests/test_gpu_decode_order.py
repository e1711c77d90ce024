"""Which decode steps hand their sequences out by length (decode_first_by_length, decode.hip), and that the order, by the
longest sequence present, does not show in the results: caches, block tables and packed keys far larger than their sequences."""
from __future__ import annotations

import random

import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HKV = 8
PLAIN = 32  # sequences of 8 kv heads that 256 workgroups take


def _by_length():
    ran = _lib.lib().dk_last_kernels()
    assert ran.startswith(b"decode_partial_kernel")
    return b"sequences by length" in ran


@pytest.mark.parametrize("form", ["paged", "packed", "cache"])
@pytest.mark.parametrize("batch,longest", [(33, 1), (48, 500), (64, 3000), (100, 900), (128, 65)])
def test_capacity_beyond_the_sequences(form, batch, longest):
    D, cap = 64, 16384
    rng = random.Random(batch)
    lens = [rng.randint(1, longest) for _ in range(batch)]
    lens[batch // 2] = longest
    g = torch.Generator(device=DEV).manual_seed(batch)
    mod = LocalStrideSparseAttention(16, cap, 64, 16, 8, num_kv_heads=HKV).to(DEV)
    q, k, v = (torch.randn(batch, n, h, D, generator=g, device=DEV, dtype=torch.bfloat16)
               for n, h in ((1, 16), (longest, HKV), (longest, HKV)))
    pages = -(-longest // 16)
    pools = [torch.nn.functional.pad(x, (0, 0, 0, 0, 0, pages * 16 - longest)).reshape(batch * pages, 16, HKV, D) for x in (k, v)]

    def step(rows):
        n, at = torch.tensor([lens[i] for i in rows], dtype=torch.int32, device=DEV), torch.tensor(rows, device=DEV)
        if form == "paged":
            table = torch.zeros(len(rows), cap // 16, dtype=torch.int32, device=DEV)
            table[:, :pages] = at[:, None] * pages + torch.arange(pages, device=DEV)
            return mod.paged_decode(q[at, 0], *pools, table, n, D ** -0.5)
        if form == "packed":
            cu = torch.nn.functional.pad(n.cumsum(0), (1, 0)).to(torch.int32)
            return mod(q[at, 0], *(torch.cat([x[i, :lens[i]] for i in rows]) for x in (k, v)), D ** -0.5, cu_seqlen_k=cu)
        wide = [torch.nn.functional.pad(x[at], (0, 0, 0, 0, 0, 5000 - longest)) for x in (k, v)]
        return mod(q[at], *wide, D ** -0.5, seqlens=n)[:, 0]

    out = step(list(range(batch)))
    assert _by_length()
    for i in range(0, batch, PLAIN):
        ref = step([min(j, batch - 1) for j in range(i, i + PLAIN)])
        assert not _by_length()
        assert torch.equal(out[i:i + PLAIN], ref[:min(PLAIN, batch - i)])


@pytest.mark.parametrize("batch,length,local,vert,D,ranked", [
    (48, 1216, 16, 64, 64, True),    # 19 blocks, rows of 17: they grow with their sequences, 17 x 64 = 1088
    (48, 1216, 8, 64, 64, False),    # rows of 9: a window and a column
    (48, 1152, 8, 64, 64, True),     # of 18 blocks
    (40, 200, 2, 8, 256, True),      # 256 dims: always
    (48, 384, 16, 8, 64, True),      # 6 blocks of 64 dims: 384
    (48, 320, 16, 8, 64, False),     # 5: 320
    (48, 4096, 13, 8, 64, True),     # rows of 20: 1280
    (48, 4096, 12, 8, 64, False),    # of 19
    (16, 1024, 16, 8, 128, False),   # growing rows of 16, 256 workgroups
    (20, 1024, 16, 8, 128, True),    # 320, two a row: 1024 each
    (10, 1536, 16, 3, 128, False),   # four a row of 19: 608
    (128, 4096, 16, 8, 128, True),   # 1024 workgroups
    (129, 4096, 16, 8, 128, False)])
def test_which_steps_take_it(batch, length, local, vert, D, ranked):
    mod = LocalStrideSparseAttention(16, length, 64, local, vert, num_kv_heads=HKV).to(DEV)
    q, k, v = (torch.randn(batch, n, h, D, device=DEV, dtype=torch.bfloat16) for n, h in ((1, 16), (length, HKV), (length, HKV)))
    mod(q, k, v, 0.1, seqlens=torch.full((batch,), length, dtype=torch.int32, device=DEV))
    assert _by_length() == ranked, mod.lut_max_row
