"""Decode steps of more than 256 workgroups hand the sequences out by length (sequence_by_length, decode.hip).
Which place takes which sequence must not show: every sequence is computed once, bit for bit as in a step whose
sequences are taken in the batch's order (256 workgroups)."""
from __future__ import annotations

import random

import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
LMAX, HQ, HKV, D = 1200, 16, 8, 64
PLAIN = 32  # sequences of 8 kv heads that 256 workgroups take


def _lengths(kind, batch):
    rng = random.Random(batch)
    if kind == "equal":
        return [777] * batch
    if kind == "ends":  # the shortest and the longest there are, many ties
        return [rng.choice((1, 63, 64, 65, LMAX - 1, LMAX)) for _ in range(batch)]
    return [rng.randint(1, LMAX) for _ in range(batch)]


@pytest.mark.parametrize("padding", ["left", "right", "packed"])
@pytest.mark.parametrize("kind", ["random", "ends", "equal"])
@pytest.mark.parametrize("batch", [33, 63, 64, 65, 100, 128, 129])  # one and two sequences a lane, and more
def test_every_sequence_as_in_the_order_of_the_batch(batch, kind, padding):
    lens = _lengths(kind, batch)
    g = torch.Generator(device=DEV).manual_seed(batch)
    q, k, v = (torch.randn(batch, n, h, D, generator=g, device=DEV, dtype=torch.bfloat16)
               for n, h in ((1, HQ), (LMAX, HKV), (LMAX, HKV)))
    mod = LocalStrideSparseAttention(HQ, LMAX, 64, 16, 4, num_kv_heads=HKV).to(DEV)  # (rows that grow with their sequences)

    def step(rows):
        n = torch.tensor([lens[i] for i in rows], dtype=torch.int32, device=DEV)
        lengths = {"left_paddings": LMAX - n} if padding == "left" else {"seqlens": n}
        at = torch.tensor(rows, device=DEV)
        if padding == "packed":
            cu = torch.nn.functional.pad(n.cumsum(0), (1, 0)).to(torch.int32)
            kp, vp = (torch.cat([x[i, :lens[i]] for i in rows]) for x in (k, v))
            return mod(q[at, 0], kp, vp, D ** -0.5, return_lse=True, cu_seqlen_k=cu)
        return mod(q[at], k[at], v[at], D ** -0.5, return_lse=True, **lengths)

    out, lse = step(list(range(batch)))
    assert (b"sequences by length" in _lib.lib().dk_last_kernels()) == (batch <= 128)
    for i in range(0, batch, PLAIN):
        rows = [min(j, batch - 1) for j in range(i, i + PLAIN)]
        ref_out, ref_lse = step(rows)
        n = min(PLAIN, batch - i)
        assert torch.isfinite(ref_out).all() and torch.isfinite(ref_lse).all()
        assert torch.equal(out[i:i + n], ref_out[:n])
        if padding == "packed":  # (heads, sequences)
            assert torch.equal(lse[:, i:i + n], ref_lse[:, :n])
        else:
            assert torch.equal(lse[i:i + n], ref_lse[:n])
