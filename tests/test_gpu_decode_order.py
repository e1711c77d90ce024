"""Decode steps that hand their sequences out by length (sequence_by_length, decode.hip): that the order, by the
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
