"""The forward kernel that small launches run, split along the keys of a row (csrc/fwd_split.h): the
sizes where it can go wrong - one token, the edges of its 32-row tiles and 32-key half blocks, rows of
fewer half blocks than waves, every tile width and padded head dims, masked tiles, more keys than
queries, packed and padded sequences, the last size before the other kernel takes over and the first
one after - against the fp32 oracle at the 16-bit bar."""
import math

import pytest
import torch

from dkernel_amd import LocalStrideSparseAttention, _lib
from helpers import LSE_TOL, TOL, assert_close, expand_heads, make_qkv, oracle_fwd
from oracle import attention as OA
from oracle import layout as OL

pytestmark = pytest.mark.gpu
DEV = "cuda"
New = LocalStrideSparseAttention.__wrapped__


def _split_ran():
    return _lib.lib().dk_last_kernels().startswith(b"mfma_fwd_split_kernel")


@pytest.mark.parametrize("B,Hq,Hkv,Lq,Lk,D,bs,dtype,causal", [
    (1, 2, 1, 2, 2, 128, 64, torch.bfloat16, True),
    (2, 2, 2, 31, 31, 64, 64, torch.float16, True),
    (1, 4, 1, 32, 32, 128, 64, torch.bfloat16, True),
    (1, 3, 1, 33, 33, 96, 64, torch.bfloat16, True),
    (1, 4, 2, 65, 65, 256, 64, torch.float16, True),
    (1, 2, 2, 97, 161, 40, 64, torch.bfloat16, True),     # the queries are the last positions, mid-tile
    (1, 8, 2, 333, 333, 128, 64, torch.bfloat16, True),
    (2, 2, 2, 200, 200, 128, 32, torch.bfloat16, True),   # masked tiles
    (1, 2, 1, 130, 130, 72, 16, torch.float16, True),
    (1, 2, 2, 300, 300, 192, 32, torch.bfloat16, True),
    (1, 4, 4, 256, 256, 64, 128, torch.float16, True),    # split tables
    (1, 4, 2, 300, 300, 128, 64, torch.bfloat16, False),
    (1, 8, 8, 2048, 2048, 128, 64, torch.bfloat16, True),  # 512 workgroups: the last launch that is split
    (1, 8, 8, 2049, 2049, 128, 64, torch.bfloat16, True),
])
def test_against_the_oracle(B, Hq, Hkv, Lq, Lk, D, bs, dtype, causal):
    print(f"case B={B} Hq={Hq} Hkv={Hkv} Lq={Lq} Lk={Lk} D={D} bs={bs} causal={causal}", flush=True)
    sm = 1 / math.sqrt(D)
    q, k, v = make_qkv(B, Lq, Lk, Hq, Hkv, D, dtype)
    step = max(bs, 64)
    Lr = (Lk + step - 1) // step * step
    bm = expand_heads(OL.block_mask(Hq, Lr, bs, 2, 3, num_kv_heads=Hkv, causal=causal), Hq)
    ro, rl = oracle_fwd(q.float(), k.float(), v.float(), bm, bs, sm, causal=causal)
    mod = New(Hq, Lr, bs, 2, 3, num_kv_heads=Hkv, causal=causal).to(DEV)
    out, lse = mod(q.to(DEV), k.to(DEV), v.to(DEV), sm, return_lse=True)
    assert _split_ran() == (Lq <= 2048), _lib.lib().dk_last_kernels()
    assert_close("O", out, ro, **TOL)
    assert_close("LSE", lse, rl, atol=LSE_TOL, rtol=0)


@pytest.mark.parametrize("D,bs", [(128, 64), (64, 32), (256, 64)])
def test_padded_and_packed(D, bs):
    print(f"case D={D} bs={bs}", flush=True)
    Hq, Hkv, Lmax, lens = 2, 1, 256, [256, 1, 100, 33]
    sm = 1 / math.sqrt(D)
    q, k, v = make_qkv(len(lens), Lmax, Lmax, Hq, Hkv, D, torch.bfloat16)
    bm = OL.block_mask(Hq, Lmax, bs, 2, 3, num_kv_heads=Hkv)
    mod = New(Hq, Lmax, bs, 2, 3, num_kv_heads=Hkv).to(DEV)
    dev = [x.to(DEV) for x in (q, k, v)]
    left = mod(*dev, sm, left_paddings=torch.tensor([Lmax - n for n in lens], dtype=torch.int32, device=DEV))
    assert _split_ran()
    right, lse = mod(*dev, sm, seqlens=torch.tensor(lens, dtype=torch.int32, device=DEV), return_lse=True)
    assert _split_ran()
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    packed = mod(*(torch.cat([x[i, :n] for i, n in enumerate(lens)]) for x in dev), sm, cu_seqlen_k=cu)
    assert _split_ran()
    for i, n in enumerate(lens):
        mask = torch.from_numpy(OA.sequence_token_mask(bm, bs, n, n))
        ro, rl = OA.dense_attention(*(x[i:i + 1, :n].float() for x in (q, k, v)), mask, sm)
        assert_close(f"right[{i}]", right[i, :n], ro[0], **TOL)
        assert_close(f"lse[{i}]", lse[i, :, :n], rl[0], atol=LSE_TOL, rtol=0)
        assert_close(f"packed[{i}]", packed[int(cu[i]):int(cu[i + 1])], ro[0], **TOL)
        assert (right[i, n:] == 0).all() and torch.isinf(lse[i, :, n:]).all()
        ro, _ = OA.dense_attention(*(x[i:i + 1, Lmax - n:].float() for x in (q, k, v)), mask, sm)
        assert_close(f"left[{i}]", left[i, Lmax - n:], ro[0], **TOL)
        assert (left[i, :Lmax - n] == 0).all()
